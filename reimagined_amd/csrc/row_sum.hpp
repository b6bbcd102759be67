// The in-order float sum of a row's squares by one workgroup, without the chain of K
// dependent adds: shared by the activation quantizer (quant.hip) and the straight-through
// backward's row norm (ste.hip).
//
// Reference semantics (OXN/nsos/ of vitorGgC569/reimagined): the sequential sum of
// Tensor::rmsnorm, src/tensor.cpp:3455-3492.
#pragma once
#include "common.hpp"

namespace nsosx {

// ===========================================================================
// E (8 or 16) consecutive elements per thread.  The in-order float sum S <- round(S + v_k) is a chain
// of K dependent adds (one lane walking the row from LDS: 8.8 cycles each, 4.2 us at
// K = 1024, 16 us at 4096), but inside one binade of S its rounding depends on S only
// through S's last bit: with S = 2^e + n ulp, round(S + v) - S is the same for every even n
// and the same for every odd n (ties go to the even neighbour).  So, the squares being >= 0,
// a run of elements that stays inside binade e is a pair of increments in ulps (for an even
// and an odd start), found by adding the run to 2^e and to 2^e + ulp, and runs compose:
// (a then b) adds a_p + b_{(p + a_p) & 1}.
//   1. every thread sums its squares; a scan gives each thread an estimate of S at its
//      first element, hence the binade it expects, and the element (if any) at which S
//      enters another one;
//   2. each thread runs the two additions over its elements, before (A) and after (B)
//      that element; a segmented scan composes the increments of neighbouring threads;
//   3. one wave walks the row's segments (about log2 K of them) with the true S in scalar
//      registers: an increment per run, one real float add per crossing.  The estimate
//      is never trusted: a run counts only if S starts and ends in the expected binade,
//      else (and at the row's start, or where one thread's elements cross twice) its
//      elements are added one by one.  Below the first binade S adds exactly, so zeros and
//      denormals are runs too.  A row of many segments (its sum grows by a binade every few
//      elements, or is infinite or NaN) is one chain, and so is what is left of a run after
//      kSumSteps threads one by one.  Same sum bit for bit.
// A call of 64 rows of 4096: 8.0 us, of zeros 5.2, as one chain 17.7.
// ===========================================================================
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int dpp0(int v) {  // 0 where the lane has no source
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}
constexpr int kDppShr1 = 0x111, kDppShr2 = 0x112, kDppShr4 = 0x114, kDppShr8 = 0x118;
constexpr int kDppBcast15 = 0x142, kDppBcast31 = 0x143, kDppWaveShr1 = 0x138;

// one thread's part of the row for the walk
struct SumRun {
    int d0, d1;  // composed increments of the segment up to this thread (B if it crosses)
    int r0, r1;  // this thread's own (B)
    int a0, a1;  // increments before its crossing element
    float v;     // the crossing element
    int meta;    // binade of d (8 bits), binade of a (8), index of the element (4), kind
};
constexpr int kSumCross = 1 << 20, kSumSerial = 2 << 20;
// A segment takes about as long as 64 additions of a chain (0.25 us).
constexpr int kSumSegment = 64, kSumSteps = 4;
// Up to here one chain over the row is the shorter way: its K additions take less than the runs'
// fixed part.  A call of 64 and of 1000 rows, us, as chain / runs: K 256 3.6 / 5.2, 3.8 / 5.7;
// 768 5.3 / 6.0, 5.7 / 6.8; 1024 6.1 / 6.1, 6.6 / 7.0, but one row 5.8 / 5.0.
constexpr int kSumChainK = 896;

template <int CTRL, int ROWS>
__device__ __forceinline__ void sum_scan_step(int& d0, int& d1, int& head) {
    const int p0 = dpp0<CTRL, ROWS>(d0), p1 = dpp0<CTRL, ROWS>(d1), ph = dpp0<CTRL, ROWS>(head);
    const int n0 = p0 + ((p0 & 1) ? d1 : d0);
    const int n1 = p1 + ((p1 & 1) ? d0 : d1);
    d0 = head ? d0 : n0;
    d1 = head ? d1 : n1;
    head |= ph;
}

__device__ __forceinline__ void sum_scan(int& d0, int& d1, int head) {
    sum_scan_step<kDppShr1, 0xF>(d0, d1, head);
    sum_scan_step<kDppShr2, 0xF>(d0, d1, head);
    sum_scan_step<kDppShr4, 0xF>(d0, d1, head);
    sum_scan_step<kDppShr8, 0xF>(d0, d1, head);
    sum_scan_step<kDppBcast15, 0xA>(d0, d1, head);
    sum_scan_step<kDppBcast31, 0xC>(d0, d1, head);
}

__device__ __forceinline__ int read_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// f plus s_sq[pos .. end) in order (end % 4 == 0)
__device__ __forceinline__ float sum_chain(float f, const float* s_sq, int pos, int end) {
    for (; pos & 3; ++pos) f = __fadd_rn(f, s_sq[pos]);
#pragma unroll 8
    for (; pos < end; pos += 4) {
        const float4 a = *reinterpret_cast<const float4*>(s_sq + pos);
        f = __fadd_rn(f, a.x);
        f = __fadd_rn(f, a.y);
        f = __fadd_rn(f, a.z);
        f = __fadd_rn(f, a.w);
    }
    return f;
}

// The in-order sum of a row's K squares (thread t's E: sq; all of them in s_sq, zeros past the
// row's end) over the first `waves` waves of the workgroup; returned to wave 0, every thread
// must call it.  K % 4 == 0.  s_run: an entry per thread; s_w, s_mask: one per wave.
template <int E>
__device__ __forceinline__ float row_sum_in_order(const float (&sq)[E], int K, int waves,
                                                  const float* s_sq, SumRun* s_run, float* s_w,
                                                  unsigned long long* s_mask) {
    if (K <= kSumChainK) {
        __syncthreads();  // s_sq
        return threadIdx.x < 64 ? sum_chain(0.0f, s_sq, 0, K) : 0.0f;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float own = 0.0f;
#pragma unroll
    for (int i = 0; i < E; i += 4) own += (sq[i] + sq[i + 1]) + (sq[i + 2] + sq[i + 3]);
    float incl = own;
    incl += __int_as_float(dpp0<kDppShr1>(__float_as_int(incl)));
    incl += __int_as_float(dpp0<kDppShr2>(__float_as_int(incl)));
    incl += __int_as_float(dpp0<kDppShr4>(__float_as_int(incl)));
    incl += __int_as_float(dpp0<kDppShr8>(__float_as_int(incl)));
    incl += __int_as_float(dpp0<kDppBcast15, 0xA>(__float_as_int(incl)));
    incl += __int_as_float(dpp0<kDppBcast31, 0xC>(__float_as_int(incl)));
    if (lane == 63) s_w[wave] = incl;
    __syncthreads();  // s_sq and the waves' sums
    float r = __int_as_float(dpp0<kDppWaveShr1>(__float_as_int(incl)));
    for (int w = 0; w < wave; ++w) r += s_w[w];

    const uint32_t kExp = 0x7f800000u;
    SumRun run;
    run.a0 = run.a1 = 0;
    run.v = 0.0f;
    const uint32_t ea = __float_as_uint(r) & kExp;
    float t0 = __uint_as_float(ea), t1 = __uint_as_float(ea | 1u);
    int crossings = 0, at = 0;
    uint32_t eb = ea;
    if (__ballot((__float_as_uint(r + own) & kExp) != ea) == 0) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
            t0 = __fadd_rn(t0, sq[i]);
            t1 = __fadd_rn(t1, sq[i]);
        }
    } else {
        float c0 = t0, c1 = t1;
#pragma unroll
        for (int i = 0; i < E; ++i) {
            r = __fadd_rn(r, sq[i]);
            const uint32_t en = __float_as_uint(r) & kExp;
            const bool cross = en != eb;
            const float n0 = __fadd_rn(t0, sq[i]), n1 = __fadd_rn(t1, sq[i]);
            c0 = cross ? t0 : c0;
            c1 = cross ? t1 : c1;
            run.v = cross ? sq[i] : run.v;
            at = cross ? i : at;
            crossings += cross ? 1 : 0;
            t0 = cross ? __uint_as_float(en) : n0;
            t1 = cross ? __uint_as_float(en | 1u) : n1;
            eb = en;
        }
        if (crossings) {
            run.a0 = (int)(__float_as_uint(c0) - ea);
            run.a1 = (int)(__float_as_uint(c1) - (ea | 1u));
        }
    }
    run.d0 = (int)(__float_as_uint(t0) - eb);
    run.d1 = (int)(__float_as_uint(t1) - (eb | 1u));
    // threads whose elements are added one by one: the first step out of zero (or the denormals), a binade with no
    // successor, two crossings, or an estimate that disagrees with the thread before
    const uint32_t before = (uint32_t)dpp0<kDppWaveShr1>((int)eb);
    const bool serial = (ea == 0u && eb != 0u) || eb >= (0xfeu << 23) || crossings > 1 || (lane > 0 && before != ea);
    if (serial) run.d0 = run.d1 = 0;
    run.r0 = run.d0;
    run.r1 = run.d1;
    int head = serial || crossings == 1;
    run.meta = (int)(eb >> 23) | (int)(ea >> 23) << 8 | at << 16 |
               (serial ? kSumSerial : (crossings == 1 ? kSumCross : 0));
    const unsigned long long heads = __ballot(head);
    sum_scan(run.d0, run.d1, head);
    if (wave > 0) s_run[threadIdx.x] = run;
    if (lane == 0) s_mask[wave] = heads;
    __syncthreads();
    if (wave > 0) return 0.0f;

    uint32_t s = 0;  // S's bits
    int pos = 0;     // elements added
    auto one_by_one = [&](int end) {  // at most to the end of pos's thread
        const int at = pos & ~(E - 1);
        const int lo = pos - at, hi = end - at;
        float c[E];
#pragma unroll
        for (int i = 0; i < E; i += 4) {
            const float4 a = *reinterpret_cast<const float4*>(s_sq + at + i);
            c[i] = a.x; c[i + 1] = a.y; c[i + 2] = a.z; c[i + 3] = a.w;
        }
        float f = __uint_as_float(s);
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const float n = __fadd_rn(f, c[i]);
            f = i >= lo && i < hi ? n : f;
        }
        s = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(f));
        pos = end;
    };
    auto chain = [&](int end) {
        s = (uint32_t)__builtin_amdgcn_readfirstlane(
            __float_as_int(sum_chain(__uint_as_float(s), s_sq, pos, end)));
        pos = end;
    };
    const unsigned long long masks = s_mask[lane & 7];  // (eight waves at most)
    int heads_in = lane < waves ? __builtin_popcountll(masks) : 0;
    heads_in += dpp0<kDppShr1>(heads_in);
    heads_in += dpp0<kDppShr2>(heads_in);
    heads_in += dpp0<kDppShr4>(heads_in);
    if (__builtin_expect(read_lane(heads_in, 7) * kSumSegment > K, 0)) return sum_chain(0.0f, s_sq, 0, K);
    for (int w = 0; w < waves; ++w) {
        const SumRun cur = run;
        if (w + 1 < waves) run = s_run[(w + 1) * 64 + lane];
        unsigned long long mask = (unsigned long long)(uint32_t)read_lane((int)(masks >> 32), w) << 32 |
                                  (uint32_t)read_lane((int)masks, w);
        const int first = w * 64;
        // the run of threads [from, to) of this wave, composed from its head
        auto advance = [&](int from, int to) {
            const uint32_t e = (uint32_t)read_lane(cur.meta, to - 1) & 0xffu;
            const uint32_t whole = s + (uint32_t)((s & 1u) ? read_lane(cur.d1, to - 1)
                                                           : read_lane(cur.d0, to - 1));
            if ((s >> 23) == e && (whole >> 23) == e) {
                s = whole;
                pos = (first + to) * E;
                return;
            }
            int d0 = cur.d0, d1 = cur.d1;
            for (int steps = 0;; ++steps) {
                if (__builtin_expect(steps == kSumSteps, 0)) return chain((first + to) * E);
                if ((s >> 23) == e) {
                    const uint32_t n = s + (uint32_t)((s & 1u) ? d1 : d0);  // after each thread
                    unsigned long long out = __ballot((n >> 23) != e) & (~0ull << from);
                    if (to < 64) out &= (1ull << to) - 1;
                    const int f = out ? __builtin_ctzll(out) : to;
                    if (f > from) {
                        s = (uint32_t)read_lane((int)n, f - 1);
                        pos = (first + f) * E;
                    }
                    if (f == to) return;
                    from = f;
                }
                // S is not where it was expected (a crossing an element early or late): this
                // thread's elements one by one, then the run from the next thread on
                one_by_one((first + from + 1) * E);
                if (++from == to) return;
                if ((s >> 23) == e) {
                    d0 = cur.r0;
                    d1 = cur.r1;
                    sum_scan(d0, d1, lane == from);
                }
            }
        };
        int from = 0;
        for (;;) {
            const int next = mask ? __builtin_ctzll(mask) : 64;
            if (pos < (first + next) * E) advance(from, next);
            if (next == 64) break;
            mask &= mask - 1;
            const int meta = read_lane(cur.meta, next);
            const int at_el = (first + next) * E;
            if (meta & kSumSerial) {
                one_by_one(at_el + E);
                from = next + 1;
            } else {
                const int j = at_el + ((meta >> 16) & 15);
                const uint32_t n = s + (uint32_t)((s & 1u) ? read_lane(cur.a1, next) : read_lane(cur.a0, next));
                const uint32_t e = (uint32_t)(meta >> 8) & 0xffu;
                if ((s >> 23) == e && (n >> 23) == e) {
                    const float v = __int_as_float(read_lane(__float_as_int(cur.v), next));
                    s = (uint32_t)__builtin_amdgcn_readfirstlane(
                        __float_as_int(__fadd_rn(__uint_as_float(n), v)));
                    pos = j + 1;
                } else {
                    one_by_one(j + 1);
                }
                from = next;  // its B is the head of the next run
            }
        }
    }
    return __uint_as_float(s);
}

// One row's int8 codes by a workgroup, E elements per thread (K <= E * blockDim.x, K % 8 == 0):
// with RMS the in-order sum, then the absmax of x * inv (x without RMS) as round(max|x| * inv) --
// rounding is monotonic -- and the codes with quantize_rows_vec_kernel's operations.  Codes to
// qrow, act_scale / inv to *scale_out / *inv_out (global memory or LDS; inv_out may be null).
// s_sq: E floats per thread, s_run: a SumRun per thread (both unused without RMS).
struct RowScratch {
    unsigned long long mask[8];
    float w[8], max[8], inv;
};

template <int DT, bool RMS, int E>
__device__ __forceinline__ void quantize_row_runs(const void* __restrict__ x, int64_t base, int K,
                                                  float q_max, float eps, float* s_sq, SumRun* s_run,
                                                  RowScratch& sc, int8_t* qrow, float* scale_out,
                                                  float* inv_out) {
    const int tid = threadIdx.x;
    const int waves = blockDim.x >> 6;
    float v[E];
    float m = 0.0f;
#pragma unroll
    for (int c = 0; c < E; c += 8) {
        float t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = 0.0f;
        if (tid * E + c < K) load8<DT>(x, base + tid * E + c, t);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            v[c + j] = t[j];
            m = fmaxf(m, fabsf(t[j]));
        }
    }
    m = wave_max(m);
    if ((tid & 63) == 0) sc.max[tid >> 6] = m;
    float inv = 1.0f;
    if constexpr (RMS) {
        float sq[E];
#pragma unroll
        for (int j = 0; j < E; ++j) sq[j] = __fmul_rn(v[j], v[j]);
#pragma unroll
        for (int j = 0; j < E; j += 4)
            *reinterpret_cast<float4*>(s_sq + tid * E + j) = make_float4(sq[j], sq[j + 1], sq[j + 2], sq[j + 3]);
        // (adding the zeros past the row's end leaves the sum as it is)
        const float sum = row_sum_in_order<E>(sq, K, min(waves, (K + 64 * E - 1) / (64 * E)), s_sq, s_run,
                                              sc.w, sc.mask);
        if (tid == 0) {
            const float mean = __fdiv_rn(sum, static_cast<float>(K));
            const float one = __fdiv_rn(1.0f, sqrtf(__fadd_rn(mean, eps)));
            sc.inv = one;
            if (inv_out) *inv_out = one;
        }
    }
    __syncthreads();
    if (RMS) inv = sc.inv;
    m = 0.0f;
    for (int w = 0; w < waves; ++w) m = fmaxf(m, sc.max[w]);
    // an infinite x gives inf * 0, which the absmax of the products skips
    if (RMS) m = fmaxf(0.0f, __fmul_rn(m, inv));
    const float denom = __fadd_rn(m, 1e-8f);
    const float s = __fdiv_rn(q_max, denom);
    if (tid == 0) *scale_out = __fdiv_rn(denom, q_max);
#pragma unroll
    for (int c = 0; c < E; c += 8) {
        if (tid * E + c >= K) break;
        float code[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float t = RMS ? __fmul_rn(v[c + j], inv) : v[c + j];
            code[j] = clamp127(rintf(__fmul_rn(t, s)));
        }
        uint2 out;
        out.x = pack4_i8(code[0], code[1], code[2], code[3]);
        out.y = pack4_i8(code[4], code[5], code[6], code[7]);
        *reinterpret_cast<uint2*>(qrow + tid * E + c) = out;
    }
}

// LDS bytes of the one-row-per-workgroup kernels (E = 8): the squares and a SumRun per thread.
inline unsigned row_sum_smem(int threads) {
    return threads * (8 * sizeof(float) + sizeof(SumRun));
}

}  // namespace nsosx
