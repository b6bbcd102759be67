// The selective scan as matrix products, for one A per head (Mamba-2) and wide states: prefill
// of the faithful block at d_state 32 .. 64.
//
// Reference semantics (OXN/nsos/ of vitorGgC569/reimagined): recurrence src/mamba2.cpp:2602-2675,
// causal conv src/mamba2.cpp:1056-1076, bias + SiLU 2437-2446.
//
// With a scalar decay per head and token, cum_i the running sum of delta_i * A2 in a chunk of
// L = 128 tokens and S the state before it,
//   y_i     = sum_{j <= i} (C_i . B_j) 2^(cum_i - cum_j) delta_j x_j + 2^cum_i C_i S + D x_i
//   S_after = 2^cum_L S + sum_j 2^(cum_L - cum_j) delta_j B_j x_j
// so a chunk is four matrix products per head of 64 channels.  The recurrence costs four
// vector operations per (token, channel, state), issue-bound: at 7078 tokens, 32 heads, 64
// states its local and full passes took 106 + 127 us.
//
// Precision is float32's: every operand is cut into three bf16 pieces by rounding (their sum is
// the value) and six of the nine products are added, the five small ones in sums of their own
// (error 2^-26 of the whole for what is left out).  cum is summed in double and kept as a
// pair of floats, so that the difference of two large sums keeps its digits.  A tile whose
// result is not finite is recomputed by the recurrence.
//
// Measured against the time-chunked recurrence, us: 7078 tokens in 8 sequences, 32 heads, 64
// states 265 -> 168 (bf16 371 -> 165), 32 states 173 -> 147; 8000 tokens of 16 heads, 32 states
// 156 -> 109; 300 tokens of 16 heads 47 -> 42.  It is bound by vector instructions (the conv, the
// cuts and the decays: about 3000 per wave of 32 tokens x 64 channels; the matrix cores
// are busy 15 % of the time), so batches that fill the chip with whole sequences stay on
// the recurrence (40800 tokens in 32 sequences: 684 against 753).
#include "scan_math.hpp"

namespace nsosx {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int kSsdThreads = 256;

// eight floats -> three chunks of eight bf16 pieces
__device__ __forceinline__ void cut8(const float (&v)[8], u32x4 (&piece)[3]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        float a = v[2 * p], b = v[2 * p + 1];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const uint32_t w = pack_bf16x2(a, b);
            piece[i][p] = w;
            a = __fsub_rn(a, __uint_as_float(w << 16));
            b = __fsub_rn(b, __uint_as_float(w & 0xffff0000u));
        }
    }
}

// acc + low += a . b over one 16-deep step: h h to acc, the other five products to low
__device__ __forceinline__ void mfma6(const v8bf (&a)[3], const v8bf (&b)[3], v16f& acc, v16f& low) {
#pragma unroll
    for (int d = 2; d >= 1; --d)
#pragma unroll
        for (int p = 0; p <= d; ++p)
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p], b[d - p], low, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
}

// A plane of rows of 64 elements (128 bytes) or 128 (256 bytes): 16-byte chunk c of row r,
// swizzled so that 16 rows read at one chunk cover all banks.
__device__ __forceinline__ int at64(int r, int c) { return r * 128 + ((c ^ ((r >> 1) & 7)) << 4); }
__device__ __forceinline__ int at128(int r, int c) { return r * 256 + ((c ^ (r & 15)) << 4); }

struct SsdTerms {
    float hi[kSsdChunk], lo[kSsdChunk];  // cum_i
    float dl[kSsdChunk];                 // delta_i, 0 past the chunk's end
    float w[kSsdChunk];                  // 2^(cum_L - cum_i) delta_i, or 2^cum_i
};

// delta and cum of the chunk's tokens for head h, by wave 0 (two tokens per lane); its sum of
// delta is returned there.
template <int ADT>
__device__ __forceinline__ float ssd_terms(const SsdArgs& g, int t0, int len, int h, float a2,
                                           SsdTerms& s) {
    const int lane = threadIdx.x;
    float d[2];
    double c[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int i = 2 * lane + e;
        const float v = load_act<ADT>(g.dt, (int64_t)min(t0 + i, g.T - 1) * g.H + h);
        d[e] = i < len ? softplus_sel(v) : 0.0f;
        c[e] = static_cast<double>(d[e]) * a2;
    }
    double incl = c[0] + c[1];
    double total = static_cast<double>(d[0]) + d[1];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double p = __shfl_up(incl, off);
        if (lane >= off) incl += p;
        total += __shfl_xor(total, off);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const double v = e ? incl : incl - c[1];
        s.hi[2 * lane + e] = static_cast<float>(v);
        s.lo[2 * lane + e] = static_cast<float>(v - static_cast<float>(v));
        s.dl[2 * lane + e] = d[e];
    }
    return static_cast<float>(total);
}

// x (conv + bias + SiLU, or raw) of COUNT consecutive tokens from chunk token i0, one channel:
// the loads apart from the arithmetic, so that a kernel can issue them first.
template <int ADT, int COUNT>
struct SsdX {
    typename raw_word<ADT>::type raw[COUNT + 3];
    float cw[4], cb;

    __device__ __forceinline__ void load(const SsdArgs& g, int t0, int ch, int i0) {
        const int taps = g.conv_w ? g.W : 1;
#pragma unroll
        for (int k = 0; k < 4; ++k)  // tap k of 4 looks 3 - k tokens back
            cw[k] = g.conv_w && k >= 4 - taps ? g.conv_w[(int64_t)ch * g.W + k - (4 - taps)] : 0.0f;
        cb = g.conv_w && g.conv_b ? g.conv_b[ch] : 0.0f;
#pragma unroll
        for (int i = 0; i < COUNT + 3; ++i)
            raw[i] = load_raw<ADT>(g.x, (int64_t)min(max(t0 + i0 + i - 3, 0), g.T - 1) * g.x_stride + ch);
    }
    __device__ __forceinline__ void finish(const SsdArgs& g, int t0, int len, int start, int i0,
                                           float (&out)[COUNT]) const {
        const int taps = g.conv_w ? g.W : 1;
        float v[COUNT + 3];
#pragma unroll
        for (int i = 0; i < COUNT + 3; ++i)
            v[i] = t0 + i0 + i - 3 >= start && i0 + i - 3 < len ? raw_to_f32<ADT>(raw[i]) : 0.0f;
#pragma unroll
        for (int i = 0; i < COUNT; ++i) {
            if (g.conv_w) {
                float acc = 0.0f;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k >= 4 - taps) acc = __fmaf_rn(cw[k], v[i + k], acc);
                out[i] = i0 + i < len ? silu_fast(acc + cb) : 0.0f;
            } else {
                out[i] = v[i + 3];
            }
        }
    }
};

// The chunk by the recurrence, for tiles whose products are not finite: thread = (channel,
// quarter of the states).  OUT: y from the carried state; else the end state from zero.
template <int ADT, bool OUT>
__device__ void ssd_sequential(const SsdArgs& g, int c, int t0, int len, int start, int h, float a2) {
    const int p = threadIdx.x >> 2, q = threadIdx.x & 3;
    const int ch = h * 64 + p, gn = (h * g.G) / g.H * g.N;
    const int per = g.N / 4;  // 8, 12 or 16
    float st[16];
    for (int n = 0; n < 16; ++n)
        st[n] = OUT && n < per ? g.carry[((int64_t)c * g.H * 64 + ch) * g.N + q * per + n] : 0.0f;
    for (int i = 0; i < len; ++i) {
        float xv[1];
        SsdX<ADT, 1> x;
        x.load(g, t0, ch, i);
        x.finish(g, t0, len, start, i, xv);
        const float dl = softplus_sel(load_act<ADT>(g.dt, (int64_t)(t0 + i) * g.H + h));
        const float decay = __builtin_amdgcn_exp2f(dl * a2), dx = dl * xv[0];
        const int64_t row = (int64_t)(t0 + i) * g.G * g.N + gn + q * per;
        float out = 0.0f;
        for (int n = 0; n < per; ++n) {
            st[n] = __fmaf_rn(decay, st[n], dx * load_act<ADT>(g.B, row + n));
            if (OUT) out = __fmaf_rn(st[n], load_act<ADT>(g.C, row + n), out);
        }
        if (OUT) {
            out += __shfl_xor(out, 1);
            out += __shfl_xor(out, 2);
            if (q == 0)
                store_act<ADT>(g.y, (int64_t)(t0 + i) * g.H * 64 + ch, __fmaf_rn(g.D[h], xv[0], out));
        }
    }
    if (!OUT)
        for (int n = 0; n < per; ++n)
            g.local[((int64_t)c * g.H * 64 + ch) * g.N + q * per + n] = st[n];
}

// Chunk and sequence bounds, clamped so that no offset table can send a tile out of bounds.
__device__ __forceinline__ void ssd_chunk(const SsdArgs& g, int c, int& t0, int& len, int& start) {
    t0 = min(max(g.chunk_cu[c], 0), g.T);
    len = min(min(max(g.chunk_cu[c + 1] - t0, 0), kSsdChunk), g.T - t0);
    start = g.seq_start[c];
}

// ---- a chunk's own end state: [64 channels x 64 states] = X^T [64 x 128] . (w B) [128 x 64],
// in two halves of 64 tokens; a wave 32 x 32 of it.  Grid: heads x chunks (heads
// fastest: neighbours share whole token rows).
template <int ADT>
__global__ __launch_bounds__(kSsdThreads, 2) void ssd_state_kernel(SsdArgs g) {
    __shared__ SsdTerms terms;
    __shared__ __align__(16) char s_x[3][64 * 128], s_b[3][64 * 128];
    const int h = blockIdx.x, c = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int t0, len, start;
    ssd_chunk(g, c, t0, len, start);
    const float a2 = a2_from_log(g.a_log[h]);
    const int64_t state0 = ((int64_t)c * g.H + h) * 64 * g.N;
    if (len == 0) {
        for (int i = tid; i < 64 * g.N; i += kSsdThreads) g.local[state0 + i] = 0.0f;
        if (tid < 64) g.sum_dl[((int64_t)c * g.H + h) * 64 + tid] = 0.0f;
        return;
    }
    const int ch = h * 64 + lane, gn = (h * g.G) / g.H * g.N;
    // a thread's 16 tokens of each half, channel and state `lane`: every load first
    SsdX<ADT, 16> xl[2];
    typename raw_word<ADT>::type bl[2][16];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int i0 = half * 64 + wave * 16;
        if (half * 64 >= len) continue;
        xl[half].load(g, t0, ch, i0);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            bl[half][i] = load_raw<ADT>(g.B, (int64_t)min(t0 + i0 + i, g.T - 1) * g.G * g.N + gn +
                                                 min(lane, g.N - 1));
    }
    if (wave == 0) {
        const float total = ssd_terms<ADT>(g, t0, len, h, a2, terms);
        g.sum_dl[((int64_t)c * g.H + h) * 64 + lane] = total;
    }
    __syncthreads();
    if (tid < kSsdChunk) {
        const float e = (terms.hi[kSsdChunk - 1] - terms.hi[tid]) + (terms.lo[kSsdChunk - 1] - terms.lo[tid]);
        terms.w[tid] = tid < len ? __builtin_amdgcn_exp2f(e) * terms.dl[tid] : 0.0f;
    }
    const int wm = wave >> 1, wn = wave & 1;
    const int li = lane & 31, lh = lane >> 5;
    v16f acc = {}, low = {};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (half * 64 >= len) break;
        const int i0 = half * 64 + wave * 16;
        float xv[16];
        xl[half].finish(g, t0, len, start, i0, xv);
        __syncthreads();  // terms.w; the previous half's planes are read
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float a[8], b[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                a[e] = xv[8 * k + e];
                b[e] = i0 + 8 * k + e < len && lane < g.N
                           ? raw_to_f32<ADT>(bl[half][8 * k + e]) * terms.w[i0 + 8 * k + e]
                           : 0.0f;
            }
            u32x4 piece[3];
            cut8(a, piece);
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(s_x[p] + at64(lane, 2 * wave + k)) = piece[p];
            cut8(b, piece);
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(s_b[p] + at64(lane, 2 * wave + k)) = piece[p];
        }
        __syncthreads();
        if (wn * 32 < g.N) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                v8bf a[3], b[3];
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    a[p] = *reinterpret_cast<const v8bf*>(s_x[p] + at64(32 * wm + li, 2 * ks + lh));
                    b[p] = *reinterpret_cast<const v8bf*>(s_b[p] + at64(32 * wn + li, 2 * ks + lh));
                }
                mfma6(a, b, acc, low);
            }
        }
    }
    // D layout of the 32x32 MFMA: register r of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4
    // (channel), column l % 32 (state)
    bool bad = false;
    const int n = 32 * wn + li;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float v = acc[r] + low[r];
        const int p = 32 * wm + 8 * (r >> 2) + 4 * lh + (r & 3);
        if (n < g.N) {
            bad |= !(fabsf(v) < __builtin_inff());
            g.local[state0 + (int64_t)p * g.N + n] = v;
        }
    }
    if (__syncthreads_or(bad)) ssd_sequential<ADT, false>(g, c, t0, len, start, h, a2);
}

// ---- a chunk's outputs: a wave owns 32 tokens x 64 channels.  C_i . B_j comes out of the
// MFMA as [j][i] (B the left operand), which is, lane by lane, the left operand of the next
// product once its 16 rows are taken in the order 4 (l / 32) + {0..3, 8..11}: the scores
// never leave the registers.  Grid: heads x chunks (heads
// fastest: neighbours share whole token rows).
// One row of B or C (64 states, 8 of each 16 for a lane half): the words of all four k steps,
// loaded together, and a step's pieces.
template <int ADT>
struct SsdRow {
    static constexpr int kWords = ADT == NSOSX_F32 ? 2 : 1;
    u32x4 w[4][kWords];

    __device__ __forceinline__ void load(const SsdArgs& g, const void* src, int t, int gn, int lh) {
        const char* row = static_cast<const char*>(src) +
                          ((int64_t)t * g.G * g.N + gn) * (ADT == NSOSX_F32 ? 4 : 2);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int n = min(16 * ks, g.N - 16) + 8 * lh;  // (past N: the last 16 again, cut to 0)
#pragma unroll
            for (int k = 0; k < kWords; ++k)
                w[ks][k] = *(global_u32x4*)(row + n * (ADT == NSOSX_F32 ? 4 : 2) + 16 * k);
        }
    }
    __device__ __forceinline__ void cut(const SsdArgs& g, int ks, v8bf (&out)[3]) const {
        float v[8];
        u32x4 piece[3];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t u = ADT == NSOSX_F32 ? w[ks][(e >> 2) & (kWords - 1)][e & 3]
                                                : (e & 1 ? w[ks][0][e >> 1] & 0xffff0000u : w[ks][0][e >> 1] << 16);
            v[e] = 16 * ks < g.N ? __uint_as_float(u) : 0.0f;
        }
        cut8(v, piece);
#pragma unroll
        for (int p = 0; p < 3; ++p) out[p] = __builtin_bit_cast(v8bf, piece[p]);
    }
};

template <int ADT>
__global__ __launch_bounds__(kSsdThreads, 2) void ssd_output_kernel(SsdArgs g) {
    extern __shared__ __align__(16) char smem_ssd[];
    __shared__ SsdTerms terms;
    char* s_x = smem_ssd;                 // 3 planes [64 channels][128 tokens]
    char* s_s = smem_ssd + 3 * 64 * 256;  // 3 planes [64 channels][64 states]
    const int h = blockIdx.x, c = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int t0, len, start;
    ssd_chunk(g, c, t0, len, start);
    if (len == 0) return;
    const int gn = (h * g.G) / g.H * g.N;
    const int li = lane & 31, lh = lane >> 5;
    const int i0 = 32 * wave;  // the wave's first token
    SsdX<ADT, 32> xl;
    SsdRow<ADT> row;
    xl.load(g, t0, h * 64 + lane, 32 * wave);
    row.load(g, g.C, t0 + min(i0 + li, len - 1), gn, lh);
    const float a2 = a2_from_log(g.a_log[h]);
    if (wave == 0) ssd_terms<ADT>(g, t0, len, h, a2, terms);
    {
        float xv[32];
        xl.finish(g, t0, len, start, 32 * wave, xv);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float a[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) a[e] = xv[8 * k + e];
            u32x4 piece[3];
            cut8(a, piece);
#pragma unroll
            for (int p = 0; p < 3; ++p)
                *reinterpret_cast<u32x4*>(s_x + p * 64 * 256 + at128(lane, 4 * wave + k)) = piece[p];
        }
        // the state before the chunk: thread = (channel, quarter of 64 states)
        const int p = tid >> 2, q = tid & 3;
        const float* src = g.carry + (((int64_t)c * g.H + h) * 64 + p) * g.N + 16 * q;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = 0.0f;
            if (16 * q < g.N) load8<NSOSX_F32>(src, 8 * k, v);  // N % 16 == 0
            u32x4 piece[3];
            cut8(v, piece);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                *reinterpret_cast<u32x4*>(s_s + i * 64 * 128 + at64(p, 2 * q + k)) = piece[i];
        }
    }
    __syncthreads();
    bool bad = false;
    if (i0 < len) {
        v16f acc[2], low[2];
#pragma unroll
        for (int pt = 0; pt < 2; ++pt) acc[pt] = low[pt] = v16f{};
        // C_i: token i0 + li, and 2^cum_i C_i S
        v8bf cf[4][3];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            row.cut(g, ks, cf[ks]);
            if (ks == 3) row.load(g, g.B, t0 + min(li, len - 1), gn, lh);  // block 0's B rows
            if (16 * ks >= g.N) continue;
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
                v8bf b[3];
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    b[p] = *reinterpret_cast<const v8bf*>(s_s + p * 64 * 128 + at64(32 * pt + li, 2 * ks + lh));
                mfma6(cf[ks], b, acc[pt], low[pt]);
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = i0 + 8 * (r >> 2) + 4 * lh + (r & 3);
            const float e = __builtin_amdgcn_exp2f(terms.hi[i] + terms.lo[i]);
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
                acc[pt][r] *= e;
                low[pt][r] *= e;
            }
        }
        const float ci = terms.hi[i0 + li], cil = terms.lo[i0 + li];
        for (int jb = 0; jb <= wave; ++jb) {
            v16f gt = {}, gl = {};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                if (16 * ks >= g.N) continue;
                v8bf bf[3];
                row.cut(g, ks, bf);
                mfma6(bf, cf[ks], gt, gl);
            }
            if (jb < wave) row.load(g, g.B, t0 + min(32 * (jb + 1) + li, len - 1), gn, lh);
            // scores of this lane's token i0 + li against tokens 32 jb + 8 q + 4 lh + e
            float m[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int j = 32 * jb + 8 * (r >> 2) + 4 * lh + (r & 3);
                const float d = (ci - terms.hi[j]) + (cil - terms.lo[j]);
                m[r] = j <= i0 + li ? (gt[r] + gl[r]) * (__builtin_amdgcn_exp2f(d) * terms.dl[j]) : 0.0f;
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = m[8 * ks + e];
                u32x4 piece[3];
                cut8(v, piece);
                v8bf a[3];
#pragma unroll
                for (int p = 0; p < 3; ++p) a[p] = __builtin_bit_cast(v8bf, piece[p]);
#pragma unroll
                for (int pt = 0; pt < 2; ++pt) {
                    v8bf b[3];
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        const char* src = s_x + p * 64 * 256;
                        const uint2 u = *reinterpret_cast<const uint2*>(
                            src + at128(32 * pt + li, 4 * jb + 2 * ks) + 8 * lh);
                        const uint2 w = *reinterpret_cast<const uint2*>(
                            src + at128(32 * pt + li, 4 * jb + 2 * ks + 1) + 8 * lh);
                        b[p] = __builtin_bit_cast(v8bf, u32x4{u.x, u.y, w.x, w.y});
                    }
                    mfma6(a, b, acc[pt], low[pt]);
                }
            }
        }
        // + D x, x back from its pieces (their sum is exact)
        const float dk = g.D[h];
#pragma unroll
        for (int pt = 0; pt < 2; ++pt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int p = 32 * pt + li;
                float xv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 2; k >= 0; --k) {
                    const uint2 u = *reinterpret_cast<const uint2*>(s_x + k * 64 * 256 +
                                                                    at128(p, 4 * wave + q) + 8 * lh);
                    xv[0] += __uint_as_float(u.x << 16);
                    xv[1] += __uint_as_float(u.x & 0xffff0000u);
                    xv[2] += __uint_as_float(u.y << 16);
                    xv[3] += __uint_as_float(u.y & 0xffff0000u);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = i0 + 8 * q + 4 * lh + e, r = 4 * q + e;
                    if (i >= len) continue;
                    const float v = __fmaf_rn(dk, xv[e], acc[pt][r] + low[pt][r]);
                    bad |= !(fabsf(v) < __builtin_inff());
                    store_act<ADT>(g.y, (int64_t)(t0 + i) * g.H * 64 + h * 64 + p, v);
                }
            }
    }
    if (__syncthreads_or(bad)) ssd_sequential<ADT, true>(g, c, t0, len, start, h, a2);
}

void launch_ssd_states(const SsdArgs& a, int act_dtype, int chunks, hipStream_t st) {
    const dim3 grid(a.H, chunks), block(kSsdThreads);
    if (act_dtype == NSOSX_F32) hipLaunchKernelGGL((ssd_state_kernel<NSOSX_F32>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((ssd_state_kernel<NSOSX_BF16>), grid, block, 0, st, a);
}

void launch_ssd_output(const SsdArgs& a, int act_dtype, int chunks, hipStream_t st) {
    const dim3 grid(a.H, chunks), block(kSsdThreads);
    constexpr int smem = 3 * 64 * 256 + 3 * 64 * 128;  // 72 KB: two workgroups per CU
    if (act_dtype == NSOSX_F32)
        hipLaunchKernelGGL((ssd_output_kernel<NSOSX_F32>), grid, block, smem, st, a);
    else
        hipLaunchKernelGGL((ssd_output_kernel<NSOSX_BF16>), grid, block, smem, st, a);
}

}  // namespace nsosx
