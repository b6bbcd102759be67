// Internal declarations shared by the BitLinear translation units (quant.hip,
// gemv.hip, skinny.hip, gemm.hip, bitlinear.hip): the problem descriptors, the
// device helpers more than one of them uses, and each unit's host launchers.
//
// Reference semantics (OXN/nsos/ of vitorGgC569/reimagined):
//   quantization  src/bitlinear.cpp:240-291, src/bitlinear_quantize_avx2.cpp:65-103
//   RMS_PERI norm src/bitlinear.cpp:460-466, src/tensor.cpp:3455-3492
//   GEMM + affine src/bitnet_adapter_avx2.cpp:52-158
//   packed format src/bitnet_adapter.cpp:570-606
#pragma once
#include "common.hpp"
#include "mamba2_step.hpp"
#include "row_sum.hpp"

#include <algorithm>
#include <cmath>

namespace nsosx {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// A ternary GEMV / GEMM problem: packed weights [N, K] (K / 16 words per row) with
// the output affine (weight scale, optional magnitude and bias per output).
struct GemvProblem {
    const uint32_t* packed;
    const float* mag;
    const float* bias;
    float ws;
    int N;
    int K;
};

struct GemmProblem {
    const uint32_t* packed;
    const float* mag;
    const float* bias;
    float ws;
    int N;
    int K;
};

// Block tile of the LDS-staged MFMA GEMMs (n x m x k).
constexpr int kG3BN = 256, kG3BM = 128, kG3BK = 128;

// MFMA layout word -> the 16 int8 operand bytes of codes k = 0..15 in natural
// order, each 64 x its ternary value: code k is a two's-complement 2-bit field at
// bits 8 (k % 4) + 6 - 2 (k / 4), so dword s (codes 4s .. 4s+3) is the word
// shifted left by 2s with all but the top two bits of every byte cleared.  The
// accumulators come out 64 x the true sums (exact in int32 for K < 2^18 / 127).
constexpr int kMfmaLayoutMaxK = 2147483647 / (64 * 127);  // 64 * 127 * K fits int32
__device__ __forceinline__ v4i unpack_word_mfma(uint32_t w) {
    return v4i{(int)(w & 0xC0C0C0C0u), (int)((w << 2) & 0xC0C0C0C0u), (int)((w << 4) & 0xC0C0C0C0u),
               (int)((w << 6) & 0xC0C0C0C0u)};
}

// Longest row that a workgroup quantizes by itself (quantize_row_runs).
constexpr int kQSmallMaxK = 4096;

// A group of a grouped GEMV with M >= 2 rows that the skinny MFMA body takes:
// K = 1024 or 2048 (its fragments fit the launch's 64 KB of LDS) and whole
// 4-output vectors (N % 4 == 0, 16-byte aligned rows).
__device__ __forceinline__ bool skinny_group(const nsosx_linear_view& v, const void* yb) {
    return (v.inputs == 1024 || v.inputs == 2048) && (v.outputs & 3) == 0 &&
           (reinterpret_cast<uintptr_t>(yb) & 15) == 0;
}

// ---- host launchers (each defined in the unit named) ----------------------
// quant.hip: RMS_PERI (when rms_input) and the int8 codes of x [M, K]
int launch_quantize_dt(const void* x, int dtype, int M, int K, int bits, int rms_input, int8_t* q,
                       float* act_scale, float* rms_ws, hipStream_t st);
// gemv.hip: the VALU GEMV (M <= 8) on the reference words
void launch_gemv(const GemvProblem& pb, const int8_t* q, const float* as, int M, void* y,
                 int y_dtype, int32_t* acc, hipStream_t st);
// gemv.hip: quantization and GEMV of one row in one launch (K % 64 == 0, K <= kQSmallMaxK)
void launch_bitlinear_row(const GemvProblem& pb, const void* x, int dtype, float q_max, bool rms,
                          int8_t* q, float* act_scale, float* rms_inv, void* y, int y_dtype,
                          hipStream_t st);
// skinny.hip: the MFMA decode GEMV (2 <= M <= 32, skinny_ok), on the reference words
// or (mfma_layout) the MFMA-layout words; and the grouped form for nsosx_grouped_gemv
bool skinny_ok(int M, int K, int N);
void launch_skinny(const GemvProblem& pb, const int8_t* q, const float* as, int M, void* y,
                   int y_dtype, int32_t* acc, bool mfma_layout, hipStream_t st);
void launch_grouped_skinny(dim3 grid, const nsosx_linear_view* views, const int8_t* q,
                           int64_t q_stride, const float* act_scale, int64_t scale_stride, int M,
                           void* y, int64_t y_stride, int y_dtype, hipStream_t st);
// gemm_small.hip: outputs too small for the 256 x 128 tiles (K % 128 == 0), on either layout;
// false where those are the faster ones (nothing launched).  kSmallMaxN: up to here the
// small tiles also beat the skinny kernel and, but for few rows of a long K, the GEMV at 2 .. 32
// rows (4 rows of K 1024 / 2048 / 4096, N 4096 / 8192 / 4096: 3.3 / 3.8 / 4.8 us against 3.9 / 6.1 /
// 10.4; with the weights from HBM 3.9 / 4.7 / 5.8 against 4.0 / 6.8 / 10.7; N 16384, K 4096 from
// HBM 8.4 against 12.2).  The stacked matrices of a decode sweep, far wider, stay with the skinny
// kernel and its four times smaller load traffic.
constexpr int kSmallMaxN = 16384;
bool launch_gemm_small(const GemmProblem& pb, const int8_t* q, const float* as, int M, void* y,
                       int y_dtype, int32_t* acc, bool mfma_layout, hipStream_t st);
// the experts' row segments, MFMA layout (perm null: rows already in slot order);
// split: whether the tiled launch would be the one with a split tail
bool launch_grouped_gemm_small(const nsosx_linear_view* views, int experts, const int32_t* offsets,
                               const int32_t* perm, const int8_t* q, const float* as, int K, int N,
                               int total_rows, int sqrelu, void* y, int y_dtype, bool split,
                               hipStream_t st);
// gemm.hip: the MFMA GEMMs on the reference words and on the MFMA layout
void launch_gemm(const GemmProblem& pb, const int8_t* q, const float* as, int M, void* y,
                 int y_dtype, int32_t* acc, hipStream_t st);
void launch_gemm_mfma(const GemmProblem& pb, const int8_t* q, const float* as, int M, void* y,
                      int y_dtype, int32_t* acc, hipStream_t st);

}  // namespace nsosx
