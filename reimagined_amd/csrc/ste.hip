// The packed BitLinear straight-through backward (src/bitlinear.cpp:1191-1357 of
// vitorGgC569/reimagined, OXN/nsos/): dW, dx, the magnitude and bias gradients.
//
// Both contractions have one f32 operand (the gradient) and one operand that bf16
// holds exactly: the int8 codes (|q| <= 127, 7 bits) and the ternary weights.  The
// f32 operand is cut into three bf16 pieces (8 + 8 + 8 significant bits: their sum
// is the value, of denormals too, since 2^24 times the operand is cut: the matrix cores
// read a denormal bf16 as zero), so three v_mfma_f32_32x32x16_bf16 with f32 accumulation give the
// products that v_mfma_f32_32x32x2_f32 gives, each exact before it is added, at a
// sixteenth of the matrix-core time per pass.  Before: two fp32-MFMA GEMMs at the
// card's fp32 rate (400 + 407 us at M = 4096, K = 1024, N = 4096), a full ternary
// GEMM for dmag (27 us) and a column reduction over two [M, N] arrays (145 us).  Now one
// launch of 230 us (200 where it runs alone) for both contractions and the column sums (MFMA issue
// alone: 94 us at the ~2.1 GHz it runs at; dW's strided gradient reads and its epilogue make its
// tiles the longer ones), a forward and backward step 1059 -> 268 us.
#include "row_sum.hpp"

#include <algorithm>
#include <cmath>

namespace nsosx {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int kTR = 128, kTC = 256;           // output tile: gradient rows x exact columns
constexpr int kTK = 32;                       // reduction depth of one LDS stage
constexpr int kSteThreads = 512;              // eight waves of 64 x 64, 2 x 4
constexpr int kPlane = kTR * kTK * 2;         // bytes of one gradient piece of a stage
constexpr int kSteStage = 3 * kPlane + kTC * kTK * 2;
constexpr int kSteSmem = 2 * kSteStage;       // double buffered: 80 KB

// The gradient operand is cut at 2^24 times its value, where the last bit of the smallest
// float (2^-149) is a normal bf16; the sums are taken back by as much.
constexpr float kSteUp = 16777216.0f;

struct SteArgs {
    const float* grad;       // [M, N]
    const float* mag;        // [N] or null
    const float* as;         // [M]
    const float* as_up;      // [M]: as * kSteUp
    const float* mag_up;     // [N]: mag * kSteUp
    const uint16_t* qT;      // bf16 [K][Mp]: the codes, reduction-contiguous, zero past M
    const uint16_t* tT;      // bf16 [K][Np]: the ternary weights, zero past N
    const uint32_t* packed;  // [N, K / 16]
    const float* wlat;       // [N, K]
    float* dW;               // [N, K]
    float* dact;             // [M, K]
    float* part_mag;         // [4 * K tiles][N] or null
    float* dbias;            // [N] or null
    float ws, clip;
    int M, K, N, Mp, Np;
    int first;               // tile of the launch's first workgroup
};

// 16-byte chunk c (8 reduction elements) of tile row r: swizzled so that the 16 rows
// a fragment read serves per clock cover all 64 banks.
__device__ __forceinline__ int tile_at(int r, int c) { return r * 64 + ((c ^ ((r >> 2) & 3)) << 4); }

// Two floats -> three pairs of bf16 pieces, by truncation: hi holds the top
// 8 significant bits, the remainders are exact.  GUARD: an infinity goes whole into hi
// (its remainder would be NaN).  A NaN stays one in every piece (the hardware's NaNs
// are quiet).
template <bool GUARD>
__device__ __forceinline__ void split3_pair(float x0, float x1, uint32_t& hi, uint32_t& mid,
                                            uint32_t& lo) {
    float r0 = __fsub_rn(x0, __uint_as_float(__float_as_uint(x0) & 0xffff0000u));
    float r1 = __fsub_rn(x1, __uint_as_float(__float_as_uint(x1) & 0xffff0000u));
    if (GUARD && fabsf(x0) == __builtin_inff()) r0 = 0.0f;
    if (GUARD && fabsf(x1) == __builtin_inff()) r1 = 0.0f;
    const float l0 = __fsub_rn(r0, __uint_as_float(__float_as_uint(r0) & 0xffff0000u));
    const float l1 = __fsub_rn(r1, __uint_as_float(__float_as_uint(r1) & 0xffff0000u));
    hi = __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
    mid = __builtin_amdgcn_perm(__float_as_uint(r1), __float_as_uint(r0), 0x07060302u);
    lo = __builtin_amdgcn_perm(__float_as_uint(l1), __float_as_uint(l0), 0x07060302u);
}

// One 128 x 256 output tile: total[rows][cols] = sum over the reduction of the gradient
// operand (rows o0 .. of dW's j or d_act's m) and the exact operand bT (columns k0 ..).
// DW: the gradient is read [reduction][output] (grad columns j, scaled by as[i]); else
// [output][reduction] (grad rows m, scaled by mag[j]).  A thread cuts 8 reduction
// elements of one tile row per stage.  The whole stages run branch-free (rows and columns
// past the operands re-read the last: their outputs are never stored), the split's VALU
// between the MFMAs and the loads two stages ahead; a last stage cut by the reduction's
// end goes through slow_stage().  So does, from the start and without the factor 2^24, a tile
// with an output that is not finite: an operand was not, or only the factor overflowed.
// colsum (DW): the thread's share of sum_i grad[i][j] for its column.
template <bool DW, bool MAG>
__device__ __forceinline__ void ste_tile(const SteArgs& g, int o0, int k0, char* smem,
                                         v16f (&total)[2][2], float& colsum) {
    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int n = 0; n < 2; ++n) acc[i][n] = total[i][n] = v16f{};
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int red = DW ? g.M : g.N;
    const int full = red / kTK;
    const uint16_t* bT = DW ? g.qT : g.tT;
    const int ldb = DW ? g.Mp : g.Np;
    // exact operand: columns tid / 4 and + 128, chunk tid % 4
    const uint16_t* bsrc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        bsrc[i] = bT + (int64_t)min(k0 + (tid >> 2) + 128 * i, g.K - 1) * ldb + (tid & 3) * 8;
    // gradient: DW column tid % 128, reduction chunk tid / 128 (the same for a whole wave);
    // else row tid / 4, chunk tid % 4
    const int row = DW ? tid & 127 : tid >> 2;
    const int chunk = DW ? wave >> 1 : tid & 3;
    const int orow = min(o0 + row, (DW ? g.N : g.M) - 1);
    const float* asrc = DW ? g.grad + orow : g.grad + (int64_t)orow * g.N;

    struct Stage {
        float f[8], sc[8];
        u32x4 b[2];
    };
    auto load = [&](int st, Stage& s) {
        const int r0 = min(st, full - 1) * kTK;  // (past the end: the last again, not used)
#pragma unroll
        for (int i = 0; i < 2; ++i) s.b[i] = *reinterpret_cast<const u32x4*>(bsrc[i] + r0);
        const int n = r0 + chunk * 8;
        if constexpr (DW) {
            const float* p = asrc + (int64_t)n * g.N;
#pragma unroll
            for (int e = 0; e < 8; ++e) s.f[e] = p[(int64_t)e * g.N];
            __builtin_memcpy(s.sc, g.as_up + n, 32);  // (4-byte aligned)
        } else {
            __builtin_memcpy(s.f, asrc + n, 32);
            if (MAG) __builtin_memcpy(s.sc, g.mag_up + n, 32);
        }
    };
    const int a_at = tile_at(row, chunk);
    auto put = [&](char* dst, const u32x4 (&piece)[3]) {
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(dst + p * kPlane + a_at) = piece[p];
    };
    auto put_b = [&](char* dst, const Stage& s) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            *reinterpret_cast<u32x4*>(dst + 3 * kPlane + tile_at((tid >> 2) + 128 * i, tid & 3)) = s.b[i];
    };
    auto cut = [&](const Stage& s, int p, u32x4 (&piece)[3]) {  // elements 2p, 2p + 1
        const float v0 = __fmul_rn(s.f[2 * p], DW || MAG ? s.sc[2 * p] : kSteUp);
        const float v1 = __fmul_rn(s.f[2 * p + 1], DW || MAG ? s.sc[2 * p + 1] : kSteUp);
        uint32_t h, m, l;
        split3_pair<false>(v0, v1, h, m, l);
        piece[0][p] = h; piece[1][p] = m; piece[2][p] = l;
    };
    auto add_cols = [&](const Stage& s, bool on) {
        const float t = ((s.f[0] + s.f[1]) + (s.f[2] + s.f[3])) + ((s.f[4] + s.f[5]) + (s.f[6] + s.f[7]));
        colsum += on ? t : 0.0f;
    };
    const int wm = wave >> 2, wn = wave & 3;
    const int li = lane & 31, lh = lane >> 5;
    // A stage is six steps of four MFMAs: two 16-deep k steps x three pieces, the smallest
    // first; fragment a(step) of the pieces, b(k step) of the exact operand.
    auto frag_b = [&](const char* s, int ks, v8bf (&b)[2]) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
            b[n] = *reinterpret_cast<const v8bf*>(s + 3 * kPlane +
                                                  tile_at(wn * 64 + n * 32 + li, 2 * ks + lh));
    };
    auto frag_a = [&](const char* s, int step, v8bf (&a)[2]) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
            a[m] = *reinterpret_cast<const v8bf*>(
                s + (2 - step % 3) * kPlane + tile_at(wm * 64 + m * 32 + li, 2 * (step / 3) + lh));
    };
    auto mfma4 = [&](const v8bf (&a)[2], const v8bf (&b)[2]) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n)
                acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[m], b[n], acc[m][n], 0, 0, 0);
    };
    // a step's fragment reads, then its MFMAs with VALU work in their shadow (left alone the
    // compiler clusters the MFMAs behind single reads and the cuts before them)
    auto fence = [&]() {
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // LDS reads
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);  // VALU
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Stage st from LDS, its first fragments already in a[0], b[0]; meanwhile stage st + 1 (in
    // s) is cut and written, and s reloaded.  The barrier stands before the last step's
    // MFMAs, whose fragments are in registers: they cover the next stage's first reads.
    v8bf a[2][2], b[2][2];
    auto advance = [&](int st, Stage& s) {
        const char* cur = smem + (st & 1) * kSteStage;
        char* nxt = smem + ((st + 1) & 1) * kSteStage;
        u32x4 piece[3];
#pragma unroll
        for (int step = 0; step < 5; ++step) {
            if (step == 1) frag_b(cur, 1, b[1]);
            frag_a(cur, step + 1, a[(step + 1) & 1]);
            mfma4(a[step & 1], b[step / 3]);
            if (step < 4) cut(s, step, piece);
            if (step == 4) {
                put(nxt, piece);
                put_b(nxt, s);
            }
            fence();
        }
        __syncthreads();
        frag_b(nxt, 0, b[0]);
        frag_a(nxt, 0, a[0]);
        mfma4(a[1], b[1]);
        if (DW) add_cols(s, st + 1 < full);
        load(st + 3, s);
        fence();
    };
    auto slow_stage = [&](int st, bool up) {  // up: times 2^24, and the columns' sums
        Stage s;
        const int n = st * kTK + chunk * 8;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int at = min(n + e, red - 1);
            const float f = asrc[DW ? (int64_t)at * g.N : (int64_t)at];
            const float sc = DW ? (up ? g.as_up : g.as)[at]
                                : (MAG ? (up ? g.mag_up : g.mag)[at] : (up ? kSteUp : 1.0f));
            s.f[e] = n + e < red ? f : 0.0f;
            v[e] = n + e < red ? __fmul_rn(f, sc) : 0.0f;
        }
        if (DW) add_cols(s, up);
#pragma unroll
        for (int i = 0; i < 2; ++i) s.b[i] = *reinterpret_cast<const u32x4*>(bsrc[i] + st * kTK);
        u32x4 piece[3];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            uint32_t h, m, l;
            split3_pair<true>(v[2 * p], v[2 * p + 1], h, m, l);
            piece[0][p] = h; piece[1][p] = m; piece[2][p] = l;
        }
        put(smem, piece);
        put_b(smem, s);
        __syncthreads();
#pragma unroll
        for (int step = 0; step < 6; ++step) {
            if (step % 3 == 0) frag_b(smem, step / 3, b[0]);
            frag_a(smem, step, a[0]);
            mfma4(a[0], b[0]);
        }
        __syncthreads();
    };

    if (full > 0) {
        Stage s0, s1;
        // (the fences keep each set's loads together, so that waiting for one set leaves the
        // other's in flight)
        load(0, s0);
        __builtin_amdgcn_sched_barrier(0);
        load(1, s1);
        __builtin_amdgcn_sched_barrier(0);
        u32x4 piece[3];
#pragma unroll
        for (int p = 0; p < 4; ++p) cut(s0, p, piece);
        put(smem, piece);
        put_b(smem, s0);
        if (DW) add_cols(s0, true);
        __builtin_amdgcn_sched_barrier(0);
        load(2, s0);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        frag_b(smem, 0, b[0]);
        frag_a(smem, 0, a[0]);
        // stage st is in LDS, st + 1 and st + 2 in s1 / s0 (in flight); a stage past the end
        // is written to the buffer that nothing reads any more
        int st = 0;
        for (; st + 1 < full; st += 2) {
            advance(st, s1);
            advance(st + 1, s0);
            // the sums of 16 stages join the total: a chain of 96 MFMA additions, not one of
            // 6 * full (4096 rows: error of dmag 6.2e-7 -> 2.5e-7 of its norm, float32 MFMA 3.0e-7)
            if ((st & 14) == 14) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        total[i][n] += acc[i][n];
                        acc[i][n] = v16f{};
                    }
            }
        }
        if (st < full) advance(st, s1);
        __syncthreads();  // (the stage past the end was read, though not used)
    }
    if (full * kTK < red) slow_stage(full, true);
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            total[i][n] = (total[i][n] + acc[i][n]) * (1.0f / kSteUp);
#pragma unroll
            for (int r = 0; r < 16; ++r) odd |= !(fabsf(total[i][n][r]) < __builtin_inff());
        }
    if (__syncthreads_or(odd)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int n = 0; n < 2; ++n) acc[i][n] = v16f{};
        for (int st = 0; st * kTK < red; ++st) slow_stage(st, false);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int n = 0; n < 2; ++n) total[i][n] = acc[i][n];
    }
}

// dW and d_act tiles in one launch (each alone is 128 tiles at 4096 x 1024, together one
// for each CU).  An XCD gets a run of consecutive tiles, K tiles fastest, so that the
// tiles sharing a gradient panel share an L2.
__global__ __launch_bounds__(kSteThreads, 2) void ste_gemm_kernel(SteArgs g) {
    extern __shared__ __align__(16) char smem_ste[];
    const int tk = (g.K + kTC - 1) / kTC;
    const int tiles_w = ((g.N + kTR - 1) / kTR) * tk;
    const int total = gridDim.x;
    const int per = total / 8;
    int t = blockIdx.x;
    if (t < per * 8) t = (t % 8) * per + t / 8;
    t += g.first;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;
    const int li = lane & 31, lh = lane >> 5;
    v16f acc[2][2];
    float colsum = 0.0f;
    const int k0 = (t < tiles_w ? t % tk : (t - tiles_w) % tk) * kTC;

    // D layout of the 32x32 MFMA: register r of lane l holds row 8 (r / 4) + 4 (l / 32) +
    // r % 4, column l % 32
    if (t >= tiles_w) {
        const int m0 = (t - tiles_w) / tk * kTR;
        if (g.mag) ste_tile<false, true>(g, m0, k0, smem_ste, acc, colsum);
        else ste_tile<false, false>(g, m0, k0, smem_ste, acc, colsum);
        const bool whole = m0 + kTR <= g.M && k0 + kTC <= g.K;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int k = k0 + wn * 64 + n * 32 + li;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                    if (whole || (m < g.M && k < g.K))
                        g.dact[(int64_t)m * g.K + k] = __fmul_rn(acc[i][n][r], g.ws);
                }
            }
        return;
    }

    const int j0 = t / tk * kTR;
    // dbias of the tile's columns: the four chunks' shares (the K tiles all read the same
    // gradient columns; the first one sums and stores)
    const bool sums = g.dbias && k0 == 0;
    ste_tile<true, false>(g, j0, k0, smem_ste, acc, colsum);
    if (sums) {
        float* s = reinterpret_cast<float*>(smem_ste);  // idle: the last stage ended in a barrier
        s[tid] = colsum;
        __syncthreads();
        if (tid < kTR && j0 + tid < g.N)
            g.dbias[j0 + tid] = ((s[tid] + s[kTR + tid]) + s[2 * kTR + tid]) + s[3 * kTR + tid];
    }
    // per 32 rows: the latent weights, the packed words and the magnitudes of the wave's
    // outputs loaded together, clamped into the matrix (each under its own branch they came
    // one at a time: 90 us of 232).  |w / clip| > 1 after rounding is |w| > clip: the next
    // float above clip already divides to more than 1 + 2^-24.
    const bool whole = j0 + kTR <= g.N && k0 + kTC <= g.K;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int jr = j0 + wm * 64 + i * 32 + 4 * lh;  // row r at + 8 (r / 4) + r % 4
        float wl[2][16], mg[16];
        uint32_t words[2][16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int j = min(jr + 8 * (r >> 2) + (r & 3), g.N - 1);
            mg[r] = g.mag ? g.mag[j] : 1.0f;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int64_t at = (int64_t)j * g.K + min(k0 + wn * 64 + n * 32 + li, g.K - 1);
                wl[n][r] = g.wlat[at];
                words[n][r] = g.part_mag ? g.packed[at >> 4] : 0u;  // K % 16 == 0
            }
        }
        float dm[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int j = jr + 8 * (r >> 2) + (r & 3);
            dm[r] = 0.0f;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int k = k0 + wn * 64 + n * 32 + li;
                const float v = acc[i][n][r];
                const uint32_t c = (words[n][r] >> (2 * (k & 15))) & 3u;
                if (k < g.K) dm[r] += c == 0u ? -v : (c == 2u ? v : 0.0f);
                const float d = fabsf(wl[n][r]) > g.clip ? 0.0f : __fmul_rn(v, mg[r]);
                if (whole || (j < g.N && k < g.K)) g.dW[(int64_t)j * g.K + k] = d;
            }
        }
        if (g.part_mag) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {  // over the 32 columns
                dm[r] += lane_xor<16>(dm[r]);
                dm[r] += lane_xor<8>(dm[r]);
                dm[r] += lane_xor<4>(dm[r]);
                dm[r] += lane_xor<2>(dm[r]);
                dm[r] += lane_xor<1>(dm[r]);
                const int j = jr + 8 * (r >> 2) + (r & 3);
                if (j < g.N && li == 0) g.part_mag[(int64_t)(4 * (k0 / kTC) + wn) * g.N + j] = dm[r];
            }
        }
    }
}

// dmag[j] = sum_i grad[i][j] * pre[i][j] with pre = acc * (as * ws), taken as
// ws * sum_k T[j][k] G[j][k] from the dW tiles' G = sum_i grad * as * q.  Where that is
// not finite, a gradient was not (0 * inf in a row's other products would leave a NaN
// in place of an infinity): the rows whose gradient (or scale) is not finite are summed from their
// own dot products, as the definition has them, by a wave per such column, up to the first NaN
// (which the sum then stays).  Gradients that overflowed everywhere, 512 x 256 x 256: 15000 us
// with a thread per column and no end at the NaN, now 66 to 104.
constexpr int kDmagCols = 32;  // columns per workgroup

__global__ __launch_bounds__(256) void ste_dmag_kernel(SteArgs g, const int8_t* __restrict__ q,
                                                       int parts, float* __restrict__ dmag) {
    __shared__ float s_sum[kDmagCols];
    const int j0 = blockIdx.x * kDmagCols;
    const int tid = threadIdx.x;
    const float inf = __builtin_inff();
    if (tid < kDmagCols) {
        const int j = j0 + tid;
        float s = 0.0f;
        if (j < g.N) {
#pragma unroll 8
            for (int c = 0; c < parts; ++c) s = __fadd_rn(s, g.part_mag[(int64_t)c * g.N + j]);
            s = __fmul_rn(s, g.ws);
            if (fabsf(s) < inf) dmag[j] = s;
        }
        s_sum[tid] = s;
    }
    __syncthreads();
    const int lane = tid & 63;
    for (int c = tid >> 6; c < kDmagCols; c += 4) {
        const float s = s_sum[c];
        if (fabsf(s) < inf) continue;
        const int j = j0 + c;
        float odd = 0.0f;
        for (int i0 = 0; i0 < g.M && odd == odd; i0 += 64) {
            const int i = min(i0 + lane, g.M - 1);
            const float gr = g.grad[(int64_t)i * g.N + j];
            const float comb = __fmul_rn(g.as[i], g.ws);
            unsigned long long rows =
                __ballot(i0 + lane < g.M && !(fabsf(gr) < inf && fabsf(comb) < inf));
            while (rows && odd == odd) {
                const int l = __builtin_ctzll(rows);
                rows &= rows - 1;
                int acc = 0;
                for (int k = 16 * lane; k < g.K; k += 16 * 64) {  // K % 16 == 0
                    const uint32_t w = g.packed[((int64_t)j * g.K + k) >> 4];
                    const int4 x = *reinterpret_cast<const int4*>(q + (int64_t)(i0 + l) * g.K + k);
                    const int xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const uint32_t code = (w >> (2 * e)) & 3u;
                        acc += (code == 0u ? -1 : (code == 2u ? 1 : 0)) *
                               static_cast<int8_t>(xs[e >> 2] >> (8 * (e & 3)));
                    }
                }
                acc = wave_sum_i32(acc);
                odd += __shfl(gr, l) * (static_cast<float>(acc) * __shfl(comb, l));
            }
        }
        // (only finite gradients: their sum overflowed, s stands)
        if (lane == 0) dmag[j] = odd != 0.0f ? odd : s;
    }
}

// A copy of an input that an output lies over.
__global__ __launch_bounds__(256) void ste_copy_kernel(const float* __restrict__ src, int64_t n,
                                                       float* __restrict__ dst) {
    for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) dst[i] = src[i];
}

// The exact operands, reduction-contiguous in bf16: qT[k][i] = q[i][k] and tT[k][j] =
// T[j][k], zero in the padding columns up to a multiple of 32.  A thread takes 16 k of
// 8 rows and writes, per k, its 8 rows as 16 bytes (a k row's 64 columns of a workgroup
// are one 128-byte line).  And the factors of the gradient operand, times kSteUp.
__global__ __launch_bounds__(256) void ste_pack_kernel(const int8_t* __restrict__ q,
                                                       const uint32_t* __restrict__ packed, int M,
                                                       int K, int N, int Mp, int Np,
                                                       uint16_t* __restrict__ qT,
                                                       uint16_t* __restrict__ tT, int qblocks,
                                                       const float* __restrict__ as,
                                                       const float* __restrict__ mag,
                                                       float* __restrict__ as_up,
                                                       float* __restrict__ mag_up) {
    const bool codes = (int)blockIdx.x < qblocks;
    const int r0 = ((codes ? blockIdx.x : blockIdx.x - qblocks) * 8 + (threadIdx.x & 7)) * 8;
    const int k0 = (blockIdx.y * 32 + (threadIdx.x >> 3)) * 16;
    const int rows = codes ? M : N, pad = codes ? Mp : Np;
    if (k0 >= K || r0 >= pad) return;  // pad % 8 == 0, K % 16 == 0
    const float* factor = codes ? as : mag;
    if (k0 == 0 && factor)
        for (int r = r0; r < min(r0 + 8, rows); ++r) (codes ? as_up : mag_up)[r] = factor[r] * kSteUp;
    uint16_t v[16][8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const bool in = r0 + r < rows;
        if (codes) {
            uint4 w = make_uint4(0u, 0u, 0u, 0u);
            if (in) w = *reinterpret_cast<const uint4*>(q + (int64_t)(r0 + r) * K + k0);
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int k = 0; k < 16; ++k)
                v[k][r] = f32_to_bf16(static_cast<float>(
                    static_cast<int8_t>((ws[k >> 2] >> (8 * (k & 3))) & 0xffu)));
        } else {
            const uint32_t w = in ? packed[((int64_t)(r0 + r) * K + k0) >> 4] : 0x55555555u;
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const uint32_t c = (w >> (2 * k)) & 3u;
                v[k][r] = c == 0u ? 0xBF80u : (c == 2u ? 0x3F80u : 0u);  // -1 / +1 / 0
            }
        }
    }
    uint16_t* dst = codes ? qT : tT;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        uint32_t w[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) w[p] = v[k][2 * p] | ((uint32_t)v[k][2 * p + 1] << 16);
        *reinterpret_cast<uint4*>(dst + (int64_t)(k0 + k) * pad + r0) =
            make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// Tensor::rmsnorm_backward (src/tensor.cpp:3997-4056) with x_norm = x * inv:
// dot = sum_k g*y / K; dx = (g - y*dot) * inv.  One wave per row.
template <int XDT>
__global__ __launch_bounds__(256) void rms_backward_kernel(const void* __restrict__ x,
                                                           const float* __restrict__ inv,
                                                           const float* __restrict__ g, int M,
                                                           int K, float* __restrict__ dx) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= M) return;
    const float s = inv[row];
    const int64_t base = (int64_t)row * K;
    float dot = 0.0f;
    for (int k = lane; k < K; k += 64) {
        const float yv = __fmul_rn(load_act<XDT>(x, base + k), s);
        dot = __fmaf_rn(g[base + k], yv, dot);
    }
    for (int off = 32; off > 0; off >>= 1) dot = __fadd_rn(dot, __shfl_xor(dot, off));
    dot = __fdiv_rn(dot, static_cast<float>(K));
    for (int k = lane; k < K; k += 64) {
        const float yv = __fmul_rn(load_act<XDT>(x, base + k), s);
        dx[base + k] = __fmul_rn(__fmaf_rn(-yv, dot, g[base + k]), s);
    }
}

// The same for rows of up to 4096 elements (K % 8 == 0), with the row's RMS on the way: a
// workgroup per row, eight elements per thread, x and the gradient read once (the two
// launches, which read x twice and the gradient twice: 9 + 20 us at 4096 x 1024).
template <int XDT>
__global__ __launch_bounds__(512) void rms_backward_row_kernel(const void* __restrict__ x, float eps,
                                                               const float* __restrict__ g, int K,
                                                               float* __restrict__ dx) {
    extern __shared__ __align__(16) float s_dyn[];
    __shared__ unsigned long long s_mask[8];
    __shared__ float s_w[8], s_dot[8], s_inv;
    const int64_t base = (int64_t)blockIdx.x * K;
    const int tid = threadIdx.x;
    const bool in = tid * 8 < K;
    float v[8], sq[8], gr[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = gr[j] = 0.0f;
    if (in) {
        load8<XDT>(x, base + tid * 8, v);
        load8<NSOSX_F32>(g, base + tid * 8, gr);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sq[j] = __fmul_rn(v[j], v[j]);
    *reinterpret_cast<float4*>(s_dyn + tid * 8) = make_float4(sq[0], sq[1], sq[2], sq[3]);
    *reinterpret_cast<float4*>(s_dyn + tid * 8 + 4) = make_float4(sq[4], sq[5], sq[6], sq[7]);
    const float sum = row_sum_in_order<8>(sq, K, blockDim.x >> 6, s_dyn, reinterpret_cast<SumRun*>(s_dyn + 8 * blockDim.x),
                                       s_w, s_mask);
    if (tid == 0)
        s_inv = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, static_cast<float>(K)), eps)));
    __syncthreads();
    const float s = s_inv;
    float dot = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        v[j] = __fmul_rn(v[j], s);
        dot = __fmaf_rn(gr[j], v[j], dot);
    }
    dot = wave_sum(dot);
    if ((tid & 63) == 0) s_dot[tid >> 6] = dot;
    __syncthreads();
    dot = 0.0f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) dot += s_dot[w];
    dot = __fdiv_rn(dot, static_cast<float>(K));
    if (!in) return;
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = __fmul_rn(__fmaf_rn(-v[j], dot, gr[j]), s);
#pragma unroll
    for (int j = 0; j < 8; ++j) dx[base + tid * 8 + j] = o[j];
}

static int64_t round256(int64_t v) { return (v + 255) & ~int64_t(255); }

// Row pitch of the transposed operands: whole stages of the reduction.
static int ste_pitch(int n) { return (n + kTK - 1) / kTK * kTK; }

struct SteWorkspace {
    uint16_t* qT;     // bf16 [K, Mp]
    uint16_t* tT;     // bf16 [K, Np]
    float* dact;      // [M, K] (rms_input only)
    float* inv;       // [M] (rms_input only)
    float* part;      // [4 * K tiles, N]
    float* grad;      // [M, N], only where an output lies over grad
    float* mag;       // [N], only where an output lies over magnitude
    float* as_up;     // [M]
    float* mag_up;    // [N]
    int Mp, Np;
    int64_t bytes;
};

static SteWorkspace ste_layout(void* base, int M, int K, int N, int rms_input) {
    SteWorkspace w{};
    w.Mp = ste_pitch(M);
    w.Np = ste_pitch(N);
    int64_t off = 0;
    auto take = [&](int64_t bytes) {
        char* p = base ? static_cast<char*>(base) + off : nullptr;
        off += round256(bytes);
        return p;
    };
    w.qT = reinterpret_cast<uint16_t*>(take(2 * (int64_t)K * w.Mp));
    w.tT = reinterpret_cast<uint16_t*>(take(2 * (int64_t)K * w.Np));
    w.dact = rms_input ? reinterpret_cast<float*>(take(4 * (int64_t)M * K)) : nullptr;
    w.inv = rms_input ? reinterpret_cast<float*>(take(4 * (int64_t)M)) : nullptr;
    w.part = reinterpret_cast<float*>(take(16 * (int64_t)((K + kTC - 1) / kTC) * N));
    w.grad = reinterpret_cast<float*>(take(4 * (int64_t)M * N));
    w.mag = reinterpret_cast<float*>(take(4 * (int64_t)N));
    w.as_up = reinterpret_cast<float*>(take(4 * (int64_t)M));
    w.mag_up = reinterpret_cast<float*>(take(4 * (int64_t)N));
    w.bytes = off;
    return w;
}

}  // namespace nsosx

using namespace nsosx;

extern "C" int64_t nsosx_bitlinear_ste_backward_workspace(int M, int K, int N, int rms_input) {
    if (M <= 0 || K <= 0 || N <= 0) return 0;
    return ste_layout(nullptr, M, K, N, rms_input).bytes;
}

extern "C" int nsosx_bitlinear_ste_backward(const void* x, int x_dtype, const int8_t* q,
                                            const float* act_scale, const float* w_latent,
                                            const uint32_t* packed, float weight_scale, int M,
                                            int K, int N, int rms_input, const float* magnitude,
                                            const float* grad, float* dx, float* dW, float* dmag,
                                            float* dbias, void* workspace, void* stream) {
    if (!q || !act_scale || !w_latent || !packed || !grad || !dx || !dW || !workspace)
        return fail(NSOSX_ERR_INVALID, "bitlinear_ste_backward: null pointer");
    if (rms_input && !x)
        return fail(NSOSX_ERR_INVALID, "bitlinear_ste_backward: rms_input needs the input x");
    if (dmag && !magnitude)
        return fail(NSOSX_ERR_INVALID, "bitlinear_ste_backward: dmag needs the magnitude");
    if (M <= 0 || K <= 0 || N <= 0)
        return fail(NSOSX_ERR_INVALID, "bitlinear_ste_backward: empty shape");
    if (K % 16 != 0 || N % 4 != 0)
        return fail(NSOSX_ERR_INVALID,
                    "bitlinear_ste_backward: K must be a multiple of 16 and N of 4");
    if (!valid_dtype(x_dtype)) return fail(NSOSX_ERR_INVALID, "bitlinear_ste_backward: bad dtype");
    if (!(weight_scale > 0.0f) || !std::isfinite(weight_scale))
        return fail(NSOSX_ERR_INVALID, "bitlinear_ste_backward: weight_scale must be finite > 0");
    if ((int64_t)M * K > ((int64_t)1 << 40) || (int64_t)M * N > ((int64_t)1 << 40) ||
        (int64_t)N * K > ((int64_t)1 << 40))
        return fail(NSOSX_ERR_OVERFLOW, "bitlinear_ste_backward: size too large");
    if (reinterpret_cast<uintptr_t>(q) % 16 || reinterpret_cast<uintptr_t>(grad) % 16 ||
        reinterpret_cast<uintptr_t>(workspace) % 256)
        return fail(NSOSX_ERR_INVALID,
                    "bitlinear_ste_backward: q and grad 16-byte, workspace 256-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const SteWorkspace ws = ste_layout(workspace, M, K, N, rms_input);
    const int tk = (K + kTC - 1) / kTC;
    const int64_t tiles = ((int64_t)(M + kTR - 1) / kTR + (N + kTR - 1) / kTR) * tk;
    const int qblocks = (ws.Mp + 63) / 64, tblocks = (ws.Np + 63) / 64;
    if (tiles > 0x7fffffff || K > 65535 * 512)
        return fail(NSOSX_ERR_OVERFLOW, "bitlinear_ste_backward: size too large");

    hipLaunchKernelGGL(ste_pack_kernel, dim3(qblocks + tblocks, (K + 511) / 512), dim3(256), 0, st,
                       q, packed, M, K, N, ws.Mp, ws.Np, ws.qT, ws.tT, qblocks, act_scale, magnitude,
                       ws.as_up, ws.mag_up);
    // The tiles of one launch store while others read.  An output over grad or magnitude makes them
    // read a copy; dx over the codes, their scales or the latent weights, which only dW's tiles
    // read, is stored by a launch after those.  (With rms_input dx is the last kernel's.)
    auto meets = [&](const void* in, int64_t bytes) {
        auto hit = [&](const float* out, int64_t n) { return out && overlaps(out, 4 * n, in, bytes); };
        return (!rms_input && hit(dx, (int64_t)M * K)) || hit(dW, (int64_t)N * K) || hit(dmag, N) ||
               hit(dbias, N);
    };
    auto copy = [&](const float* src, int64_t n, float* dst) -> const float* {
        hipLaunchKernelGGL(ste_copy_kernel, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 16384)),
                           dim3(256), 0, st, src, n, dst);
        return dst;
    };
    const float* gsrc = meets(grad, 4 * (int64_t)M * N) ? copy(grad, (int64_t)M * N, ws.grad) : grad;
    const float* msrc = magnitude && meets(magnitude, 4 * (int64_t)N) ? copy(magnitude, N, ws.mag) : magnitude;
    const bool dx_last = !rms_input && (overlaps(dx, 4 * (int64_t)M * K, q, (int64_t)M * K) ||
                                        overlaps(dx, 4 * (int64_t)M * K, act_scale, 4 * (int64_t)M) ||
                                        overlaps(dx, 4 * (int64_t)M * K, w_latent, 4 * (int64_t)N * K));

    // dW = gp^T @ (x_q * act_scale), zero where |W / (ws + 1e-8f)| > 1 (bitlinear.cpp:1293-1321),
    // with gp = grad * magnitude taken as magnitude[j] * (grad^T @ ...); d_act = gp @ (ternary *
    // weight_scale) (1340); the column sums behind dmag and dbias (1267-1290) on the way
    SteArgs g{};
    g.grad = gsrc; g.mag = msrc; g.as = act_scale; g.as_up = ws.as_up; g.mag_up = ws.mag_up; g.qT = ws.qT; g.tT = ws.tT;
    g.packed = packed; g.wlat = w_latent; g.dW = dW; g.dact = rms_input ? ws.dact : dx;
    g.part_mag = dmag ? ws.part : nullptr; g.dbias = dbias;
    g.ws = weight_scale; g.clip = weight_scale + 1e-8f;
    g.M = M; g.K = K; g.N = N; g.Mp = ws.Mp; g.Np = ws.Np;
    const int64_t tiles_w = (int64_t)(N + kTR - 1) / kTR * tk;
    hipLaunchKernelGGL(ste_gemm_kernel, dim3((unsigned)(dx_last ? tiles_w : tiles)), dim3(kSteThreads),
                       kSteSmem, st, g);
    if (dmag)
        hipLaunchKernelGGL(ste_dmag_kernel, dim3((N + kDmagCols - 1) / kDmagCols), dim3(256), 0, st, g, q,
                           4 * tk, dmag);
    if (dx_last) {
        g.first = (int)tiles_w;
        hipLaunchKernelGGL(ste_gemm_kernel, dim3((unsigned)(tiles - tiles_w)), dim3(kSteThreads), kSteSmem,
                           st, g);
    }

    // dx = rmsnorm_backward(x, d_act, x_norm) (bitlinear.cpp:1352-1355)
    if (rms_input) {
        if (K <= 4096 && reinterpret_cast<uintptr_t>(x) % 16 == 0) {  // K % 16 == 0: whole chunks
            const int threads = (K / 8 + 63) / 64 * 64;
            if (x_dtype == NSOSX_F32)
                hipLaunchKernelGGL((rms_backward_row_kernel<NSOSX_F32>), dim3(M), dim3(threads),
                                   row_sum_smem(threads), st, x, 1e-6f, ws.dact, K, dx);
            else
                hipLaunchKernelGGL((rms_backward_row_kernel<NSOSX_BF16>), dim3(M), dim3(threads),
                                   row_sum_smem(threads), st, x, 1e-6f, ws.dact, K, dx);
            return check_launch("bitlinear_ste_backward");
        }
        launch_rms_inv(x, x_dtype, M, K, 1e-6f, ws.inv, st);
        const dim3 grid((M + 3) / 4);
        if (x_dtype == NSOSX_F32)
            hipLaunchKernelGGL((rms_backward_kernel<NSOSX_F32>), grid, dim3(256), 0, st, x, ws.inv,
                               ws.dact, M, K, dx);
        else
            hipLaunchKernelGGL((rms_backward_kernel<NSOSX_BF16>), grid, dim3(256), 0, st, x,
                               ws.inv, ws.dact, M, K, dx);
    }
    return check_launch("bitlinear_ste_backward");
}
