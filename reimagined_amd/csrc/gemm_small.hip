// Ternary GEMMs whose output is too small to fill the chip with 256 x 128 tiles:
// decode batches past the skinny kernel's shapes, short prompts, and the experts of a
// routed batch of few rows.
//
// Reference semantics (OXN/nsos/ of vitorGgC569/reimagined):
//   GEMM + affine    src/bitnet_adapter_avx2.cpp:52-158
//   per-expert GEMMs src/jamba.cpp:3896-3946
#include "gemm_tiles.hpp"

namespace nsosx {

// A workgroup owns 32 NT outputs x 32 MT tokens; its four waves split K (128-deep
// blocks, a contiguous quarter each) and every wave runs v_mfma_i32_32x32x32_i8 on
// fragments read straight from memory: lane l (row l % 32, half g = l / 32) takes the
// block's 64 k values of its half, one 16-byte word group per weight row and 64
// contiguous bytes per activation row, the next block's loads in flight.  Nothing is
// staged and nothing waits between the waves until the end, where the four partial
// tiles (integers: any order, the same bits) meet in LDS and leave as whole row pieces.
// What bounds a call is one memory round trip and the waves' own loads (a 64 x 64 tile
// reads 12 KB per 16 MFMAs through the vector cache, about half the matrix rate), which
// is why the large GEMMs keep the staged kernel.
constexpr int kSmallPitchPad = 4;  // ints: a row's 16-byte pieces shift by one bank group

template <bool SWZ, int NT, int MT>
__device__ __forceinline__ void small_tile(const GemmProblem& pb, const int8_t* __restrict__ q,
                                           const float* __restrict__ act_scale,
                                           const int32_t* __restrict__ perm, int seg_begin,
                                           int seg_rows, int n0, int m0, int sqrelu, void* y,
                                           int y_bf16, int32_t* acc_out, int32_t* s_part) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, li = lane & 31;
    const int blocks = pb.K / kG3BK;
    const int b0 = blocks * wave / 4, b1 = blocks * (wave + 1) / 4;
    // rows past N or the segment re-read its last one; their outputs are not stored
    const char* wsrc[NT];
    const char* xsrc[MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
        wsrc[n] = reinterpret_cast<const char*>(pb.packed) +
                  (int64_t)min(n0 + 32 * n + li, pb.N - 1) * (pb.K / 4) + g * 16;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int slot = seg_begin + min(m0 + 32 * m + li, seg_rows - 1);
        xsrc[m] = reinterpret_cast<const char*>(q) + (int64_t)(perm ? perm[slot] : slot) * pb.K + g * 64;
    }
    u32x4 w[2][NT], x[2][MT][4];
    auto load = [&](int b, u32x4 (&wb)[NT], u32x4 (&xb)[MT][4]) {
        const int at = min(b, max(b1 - 1, 0));
#pragma unroll
        for (int n = 0; n < NT; ++n) wb[n] = *(global_u32x4*)(wsrc[n] + at * 32);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) xb[m][ks] = *(global_u32x4*)(xsrc[m] + at * 128 + ks * 16);
    };
    v16i acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = v16i{};
    auto contract = [&](const u32x4 (&wb)[NT], const u32x4 (&xb)[MT][4]) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            v4i a[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                if constexpr (SWZ) {
                    a[n] = unpack_word_mfma(wb[n][ks]);
                } else {
                    uint32_t wv[4], wt[4];
                    unpack_word(wb[n][ks], wv);
                    transpose16(wv, wt);
                    a[n] = v4i{(int)wt[0], (int)wt[1], (int)wt[2], (int)wt[3]};
                }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const v4i b = {(int)xb[m][ks][0], (int)xb[m][ks][1], (int)xb[m][ks][2], (int)xb[m][ks][3]};
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[n][m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[n], b, acc[n][m], 0, 0, 0);
            }
        }
    };
    if (b0 < b1) {
        load(b0, w[0], x[0]);
        int b = b0;
        for (; b + 1 < b1; b += 2) {
            load(b + 1, w[1], x[1]);
            contract(w[0], x[0]);
            load(b + 2, w[0], x[0]);
            contract(w[1], x[1]);
        }
        if (b < b1) contract(w[0], x[0]);
    }
    // accumulator r of a lane: output 8 (r / 4) + 4 g + r % 4 of the 32, token li
    constexpr int kPitch = 32 * NT + kSmallPitchPad;
    constexpr int kPart = 32 * MT * kPitch;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                *reinterpret_cast<int4*>(s_part + wave * kPart + (32 * m + li) * kPitch + 32 * n +
                                         8 * c + 4 * g) =
                    make_int4(acc[n][m][4 * c], acc[n][m][4 * c + 1], acc[n][m][4 * c + 2],
                              acc[n][m][4 * c + 3]);
    __syncthreads();
    // eight outputs of one token per thread and step
    for (int i = threadIdx.x; i < 32 * MT * 4 * NT; i += 256) {
        const int row = i / (4 * NT), c = i % (4 * NT);
        const int ml = m0 + row, n = n0 + 8 * c;
        if (ml >= seg_rows || n >= pb.N) continue;
        int sum[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] = 0;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int32_t* src = s_part + p * kPart + row * kPitch + 8 * c;
            const int4 u = *reinterpret_cast<const int4*>(src);
            const int4 v = *reinterpret_cast<const int4*>(src + 4);
            sum[0] += u.x; sum[1] += u.y; sum[2] += u.z; sum[3] += u.w;
            sum[4] += v.x; sum[5] += v.y; sum[6] += v.z; sum[7] += v.w;
        }
        const int64_t orow = seg_begin + ml;
        const float comb = __fmul_rn(act_scale[perm ? perm[orow] : orow], pb.ws);
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (SWZ) sum[e] >>= 6;  // the MFMA layout's operands are 64 x the ternary values
            o[e] = dequant(sum[e], comb, pb.mag, pb.bias, min(n + e, pb.N - 1));
            if (sqrelu) {
                o[e] = o[e] > 0.0f ? o[e] : 0.0f;
                o[e] = __fmul_rn(o[e], o[e]);
            }
        }
        const int64_t at = orow * pb.N + n;
        if (acc_out)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (n + e < pb.N) acc_out[at + e] = sum[e];
        if (!y) continue;
        const bool whole = n + 8 <= pb.N;
        if (y_bf16) {
            uint16_t* dst = static_cast<uint16_t*>(y) + at;
            if (whole && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
                *reinterpret_cast<uint4*>(dst) =
                    make_uint4(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]),
                               pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7]));
                continue;
            }
        } else {
            float* dst = static_cast<float*>(y) + at;
            if (whole && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
                *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
                *reinterpret_cast<float4*>(dst + 4) = make_float4(o[4], o[5], o[6], o[7]);
                continue;
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (n + e >= pb.N) break;
            if (y_bf16) static_cast<uint16_t*>(y)[at + e] = f32_to_bf16(o[e]);
            else static_cast<float*>(y)[at + e] = o[e];
        }
    }
}

template <int NT, int MT>
constexpr int small_smem() { return 4 * 32 * MT * (32 * NT + kSmallPitchPad) * 4; }

template <bool SWZ, int NT, int MT>
__global__ __launch_bounds__(256) void gemm_small_kernel(GemmProblem pb, const int8_t* __restrict__ q,
                                                         const float* __restrict__ act_scale, int M,
                                                         void* y, int y_bf16, int32_t* acc_out) {
    extern __shared__ __align__(16) int32_t smem_small[];
    int nt, mt;
    xcd_tile(blockIdx.x, (pb.N + 32 * NT - 1) / (32 * NT), (M + 32 * MT - 1) / (32 * MT), nt, mt);
    small_tile<SWZ, NT, MT>(pb, q, act_scale, nullptr, 0, M, nt * 32 * NT, mt * 32 * MT, 0, y,
                            y_bf16, acc_out, smem_small);
}

// One launch over the experts' row tiles (ceil(rows_e / 32 MT) each, found from the
// offsets), n fastest.
template <int NT, int MT>
__global__ __launch_bounds__(256) void grouped_gemm_small_kernel(
    const nsosx_linear_view* views, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ perm, const int8_t* __restrict__ q,
    const float* __restrict__ act_scale, int sqrelu, void* y, int y_bf16, int ntn, int experts) {
    extern __shared__ __align__(16) int32_t smem_small[];
    const int nt = blockIdx.x % ntn;
    int tile = blockIdx.x / ntn;
    int e = 0, seg_begin = 0, seg_rows = 0;
    for (; e < experts; ++e) {
        seg_begin = offsets[e];
        seg_rows = max(offsets[e + 1] - seg_begin, 0);
        const int tiles = (seg_rows + 32 * MT - 1) / (32 * MT);
        if (tile < tiles) break;
        tile -= tiles;
    }
    if (e == experts) return;
    const nsosx_linear_view v = views[e];
    const int n0 = nt * 32 * NT;
    if (n0 >= v.outputs) return;
    const GemmProblem pb{v.packed, v.magnitude, v.bias, v.weight_scale, v.outputs, v.inputs};
    small_tile<true, NT, MT>(pb, q, act_scale, perm, seg_begin, seg_rows, n0, tile * 32 * MT, sqrelu,
                             y, y_bf16, nullptr, smem_small);
}

// Which kernel takes a shape: the estimated time of each in 0.1 us, from a sweep of K 768 ..
// 4096, N 768 .. 16384 and 9 .. 3000 rows (weights in the caches).  A small-tile launch runs
// in rounds of 256 workgroups (one per CU; more per CU only overlap, their loads share the
// vector cache), each a term per 128-deep block of K and a fixed one; 256 of the 256 x 128 kernel's
// tiles take 0.19 us per block and 0.28 more per 32 rows that they hold.  Measured, us (small /
// 256 x 128 tiles): K 2048, N 8192: 64 rows 5.8 / 17 (and 41 on the old few-row kernel),
// 200 rows 14.5 / 17.6, 300 rows 19.6 / 17.7; K 4096, N 1024: 64 rows 7.3 / 30, 1500 rows
// 20.5 / 30.5, 3000 rows 33 / 31.  Weights from HBM add about as much to either side and leave
// the rule where it is: K 2048, N 8192: 64 rows 7.0 / 19.2, 200 rows 15.7 / 19.1; 64 routed rows over
// 8 experts, 1024 -> 4096 -> 1024: 7.4 / 9.8 up, 9.0 / 29.3 down; 256 rows 12.9 / 12.8, 16 / 38.5.
struct SmallChoice {
    int nt, mt;  // 0: the 256 x 128 kernel
};

static SmallChoice small_choice(int K, int N, double rows32, double rows64, double rows128,
                                double large_extra, double small_extra) {
    const double kb = K / kG3BK;
    const double n32 = (N + 31) / 32, n64 = (N + 63) / 64, n256 = (N + kG3BN - 1) / kG3BN;
    auto rounds = [](double tiles) { return std::ceil(tiles / 256.0); };
    const double c11 = 22 + small_extra + rounds(n32 * rows32) * (5.5 + 1.46 * kb);
    const double c21 = 22 + small_extra + rounds(n64 * rows32) * (6.0 + 1.75 * kb);
    const double c22 = 22 + small_extra + rounds(n64 * rows64) * (18.0 + 2.65 * kb);
    const double large =
        46 + std::max(8.0 * kb, n256 * kb * (1.9 * rows128 + 2.8 * rows32) / 256) + large_extra;
    const double best = std::min(std::min(c11, c21), c22);
    if (large <= best) return {0, 0};
    if (c11 == best) return {1, 1};
    return c21 == best ? SmallChoice{2, 1} : SmallChoice{2, 2};
}

template <bool SWZ>
static bool launch_small_t(const GemmProblem& pb, const int8_t* q, const float* as, int M, void* y,
                           int y_dtype, int32_t* acc, hipStream_t st) {
    const SmallChoice c = small_choice(pb.K, pb.N, (M + 31) / 32, (M + 63) / 64, (M + 127) / 128, 0, 0);
    if (c.nt == 0) return false;
    const int ybf = y_dtype == NSOSX_BF16;
#define NSOSX_SMALL(NT, MT)                                                                     \
    hipLaunchKernelGGL((gemm_small_kernel<SWZ, NT, MT>),                                        \
                       dim3(((pb.N + 32 * NT - 1) / (32 * NT)) * ((M + 32 * MT - 1) / (32 * MT))), \
                       dim3(256), (small_smem<NT, MT>()), st, pb, q, as, M, y, ybf, acc)
    if (c.nt == 1) NSOSX_SMALL(1, 1);
    else if (c.mt == 1) NSOSX_SMALL(2, 1);
    else NSOSX_SMALL(2, 2);
#undef NSOSX_SMALL
    return true;
}

bool launch_gemm_small(const GemmProblem& pb, const int8_t* q, const float* as, int M, void* y,
                       int y_dtype, int32_t* acc, bool mfma_layout, hipStream_t st) {
    if (pb.K % kG3BK != 0) return false;
    return mfma_layout ? launch_small_t<true>(pb, q, as, M, y, y_dtype, acc, st)
                       : launch_small_t<false>(pb, q, as, M, y, y_dtype, acc, st);
}

// The experts' row counts are on the device: each expert's last tile is taken as three
// quarters of a tile more than its share.  The large kernel's workgroups find their segment in 0.1 us
// per expert, and its split launch takes about 4 us and 0.45 per expert more (ws against not, 4096 x
// 512, 1000 rows: 2 experts 36.9 / 32.7, 16 40.1 / 29.1, 64 62.8 / 30.8).  The small tiles read the
// codes on every XCD, which past 8 MB (two L2s) takes its time: 5000 rows of 4096, 512 outputs,
// 8 experts 48.2 us small, 42.8 large.
bool launch_grouped_gemm_small(const nsosx_linear_view* views, int experts, const int32_t* offsets,
                               const int32_t* perm, const int8_t* q, const float* as, int K, int N,
                               int total_rows, int sqrelu, void* y, int y_dtype, bool split,
                               hipStream_t st) {
    auto tiles = [&](int rows) {
        return std::min<double>(total_rows, std::ceil((double)total_rows / rows + 0.75 * experts));
    };
    const double codes = std::max(0.0, (double)total_rows * K - 8e6) * 8e-6;  // 10 TB/s, eight XCDs
    const double large_extra = experts + (split ? 40 + 4.5 * experts : 0);
    const SmallChoice c = small_choice(K, N, tiles(32), tiles(64), tiles(128), large_extra, codes);
    if (c.nt == 0) return false;
    const int ntn = (N + 32 * c.nt - 1) / (32 * c.nt);
    // >= the real row tiles, each of which holds a row (a workgroup past them walks every expert: 2
    // rows, 64 experts, 1024 -> 4096 63 us without the bound, 7.1 with it)
    const int ntm = std::min(total_rows, (total_rows + 32 * c.mt - 1) / (32 * c.mt) + experts);
    if ((int64_t)ntn * ntm > 0x7fffffff) return false;
    const int ybf = y_dtype == NSOSX_BF16;
#define NSOSX_SMALL(NT, MT)                                                                       \
    hipLaunchKernelGGL((grouped_gemm_small_kernel<NT, MT>), dim3(ntn * ntm), dim3(256),           \
                       (small_smem<NT, MT>()), st, views, offsets, perm, q, as, sqrelu, y, ybf, ntn, \
                       experts)
    if (c.nt == 1) NSOSX_SMALL(1, 1);
    else if (c.mt == 1) NSOSX_SMALL(2, 1);
    else NSOSX_SMALL(2, 2);
#undef NSOSX_SMALL
    return true;
}

}  // namespace nsosx
