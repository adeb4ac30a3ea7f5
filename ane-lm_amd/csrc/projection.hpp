// What the projection kernels (projection.hip: few rows of x; gemm.hip: many)
// share: their arguments, epilogues and operand helpers.
#pragma once

#include "anelm_common.hpp"

namespace anelm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float r16(float v) { return (float)to_f16(v); }
// fp16 bits (low 16 of h) widened exactly
__device__ __forceinline__ float h2f_bits(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

__device__ __forceinline__ half8 to_half8(float4 a, float4 b) {
    half8 r;
    r[0] = to_f16(a.x);
    r[1] = to_f16(a.y);
    r[2] = to_f16(a.z);
    r[3] = to_f16(a.w);
    r[4] = to_f16(b.x);
    r[5] = to_f16(b.y);
    r[6] = to_f16(b.z);
    r[7] = to_f16(b.w);
    return r;
}

__device__ __forceinline__ half8 as_half8(uint4 u) {
    half8 r;
    __builtin_memcpy(&r, &u, 16);
    return r;
}

// (x * s) * gamma for four inputs, gamma as two packed bf16 pairs: the fused
// RMSNorm's output, before its fp16 rounding
__device__ __forceinline__ float4 norm_scale(float4 v, float s, uint32_t g01, uint32_t g23) {
    v.x = (v.x * s) * bf16_to_f32(g01 & 0xFFFFu);
    v.y = (v.y * s) * bf16_to_f32(g01 >> 16);
    v.z = (v.z * s) * bf16_to_f32(g23 & 0xFFFFu);
    v.w = (v.w * s) * bf16_to_f32(g23 >> 16);
    return v;
}

struct ProjArgs {
    float* y;
    const void* x;  // fp32, or fp16 already rounded (XH)
    const uint16_t* w;
    int out_dim, in_dim, batch;
    long ld_x, ld_y;
    // fused prologue (kNorm): x replaced by rmsnorm(x) * gamma, gamma bf16 [in_dim]
    const uint16_t* gamma;
    float eps;
    // SwiGLU epilogue (kSwiGLU, kSwiGLU16): the up rows follow the gate rows at this offset
    long pair_rows;
    // kSwiGLU16, kStore16: the output as fp16 bits (row stride ld_y) instead of y
    uint16_t* y16;
    // y rows 16-byte aligned (y and ld_y), for the LDS kernel's float4 stores
    bool vec_y;
};

// What the epilogue does with the rounded projection p = fp16(sum) (as fp32):
enum Epilogue {
    kStore = 0,   // y = p
    kAdd = 1,     // y = y + p  (the residual add of qwen3.cpp:516, :527)
    kSwiGLU = 2,  // y = silu(p_gate) * p_up  (core/ane_runtime.cpp:393-395)
    kSwiGLU16 = 3,  // the same rounded to fp16 (nearest even) into y16: the next projection's input
    kStore16 = 4,   // y16 = p as fp16 bits (the ANE kernels' own fp16 output)
    kSwiGLU16T = 5, // kSwiGLU16 with y16 in the tiled layout (out_dim columns): the tiled projection's input
};
constexpr bool is_swiglu(int epi) { return epi == kSwiGLU || epi == kSwiGLU16 || epi == kSwiGLU16T; }

__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
    return (uint32_t)__builtin_bit_cast(uint16_t, to_f16(lo)) | ((uint32_t)__builtin_bit_cast(uint16_t, to_f16(hi)) << 16);
}

// the forms of x (see proj_dot_kernel)
enum : int {
    kXF32 = 0,
    kXNorm = 1,
    kXF16 = 2,
};

// ---- 3 to 16 rows of x, W row-major (rows.hip)
bool rows_takes(const ProjArgs& a);
template <int XM, int EPI>
void launch_rows(const ProjArgs& a, hipStream_t st);

// ---- many rows of x (gemm.hip) -------------------------------------------------
// Whether the block-tiled kernel takes a projection of fp16 x.
bool gemm_takes(const ProjArgs& a, int epi);
// Launches it (XT / TILED: the layouts of x and W).
template <int EPI, bool TILED, bool XT>
void launch_gemm(ProjArgs a, hipStream_t st);

}  // namespace anelm
