// Per-token terms of the selective scan shared by its kernels (scan.hip, ssd.hip).
#pragma once
#include "common.hpp"

namespace nsosx {

__device__ __forceinline__ float softplus_ref(float v) {
    if (v > 20.0f) return v;
    if (v < -20.0f) return expf(v);
    return log1pf(expf(v));
}

__device__ __forceinline__ float a2_from_log(float a_log) {
    return static_cast<float>(-exp(static_cast<double>(a_log)) * 1.4426950408889634);
}

__device__ __forceinline__ float dpp_xor1(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_xor2(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));
}

// Native-instruction forms of softplus and SiLU for the per-(token, channel)
// terms (v_exp_f32 / v_log_f32 / v_rcp_f32, each about 1 ulp): log1p(e) is
// taken as log(u) * e / (u - 1) with u = 1 + e, which cancels the rounding of
// u (Kahan), so the relative error stays at a few ulp for all dt_raw.
__device__ __forceinline__ float exp_native(float v) {
    return __builtin_amdgcn_exp2f(v * 1.4426950408889634f);
}

__device__ __forceinline__ float softplus_fast(float v) {
    if (v > 20.0f) return v;
    if (v < -20.0f) return expf(v);
    const float e = exp_native(v);
    const float u = 1.0f + e;
    if (u == 1.0f) return e;
    return __builtin_amdgcn_logf(u) * 0.6931471805599453f * (e * __builtin_amdgcn_rcpf(u - 1.0f));
}

__device__ __forceinline__ float silu_fast(float v) {
    return v * __builtin_amdgcn_rcpf(1.0f + exp_native(-v));
}

// softplus_fast() without branches: the three regimes are formed and selected.
__device__ __forceinline__ float softplus_sel(float v) {
    const float e = exp_native(v);
    const float u = 1.0f + e;
    const float mid = __builtin_amdgcn_logf(u) * 0.6931471805599453f * (e * __builtin_amdgcn_rcpf(u - 1.0f));
    return v > 20.0f ? v : (u == 1.0f ? e : mid);
}

// ---- the matrix form (ssd.hip) ------------------------------------------------
struct SsdArgs {
    const void* x;
    int64_t x_stride;
    const float* conv_w;  // [D, W] or null
    const float* conv_b;
    int W;
    const void* dt;       // [T, H]
    const float* a_log;   // [H]
    const void* B;        // [T, G * N]
    const void* C;
    const float* D;       // [H]
    const int32_t* chunk_cu;   // [chunks + 1]
    const int32_t* seq_start;  // [chunks]
    float* local;         // [chunks, H * 64, N] a chunk's own end state
    float* sum_dl;        // [chunks, H * 64]
    const float* carry;   // [chunks, H * 64, N] the state before a chunk
    void* y;              // [T, H * 64]
    int T, H, N, G;
};

constexpr int kSsdChunk = 128;

// the shapes it takes: one A per head of 64 channels, N in (16, 64] a multiple of 16
inline bool ssd_shape(int S, int T, int H, int P, int N) {
    const int64_t chunks = (int64_t)S + (T + kSsdChunk - 1) / kSsdChunk;
    return P == 64 && N > 16 && N <= 64 && N % 16 == 0 && H <= 65535 && chunks <= 65535 &&
           chunks * H * P * N <= ((int64_t)1 << 28);  // 1 GiB of states
}
void launch_ssd_states(const SsdArgs& a, int act_dtype, int chunks, hipStream_t st);
void launch_ssd_output(const SsdArgs& a, int act_dtype, int chunks, hipStream_t st);

}  // namespace nsosx
