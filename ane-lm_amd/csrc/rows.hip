// The fp16 projections of projection.hip for 3 to 16 rows of x against a
// row-major W: each byte of W is used once, so they are bound by how W streams
// from HBM.
//
// One workgroup per 16 outputs (the SwiGLU: 16 gate and 16 up rows), its NW
// waves taking 128-input chunks in turn.  The MFMA operand layout wants lane l
// to hold row l%16, so loading W straight into it touches 64 bytes of each of
// 16 rows per instruction, and 64-byte pieces of a row-major matrix stream at
// 3.4-3.9 TB/s where whole 256-byte pieces reach 5-6 (50 and 100 MB read cold).
// Here a wave loads 256 bytes of each of four rows per instruction and takes
// its 16 x 128 chunk through LDS into the operand layout.  The LDS area is the
// wave's own, so its lanes need no workgroup barrier between them, only their
// writes and reads kept in order (wave_lds_sync), and its 16-byte pieces are
// placed at piece ^ row, which spreads the operand reads over the banks.  The x rows of
// the chunk go the same way: fp16 as they are, fp32 rounded (after the RMSNorm
// with kXNorm, whose scales each workgroup works out first) into the same
// places.  One chunk per wave in flight: a second one costs registers that
// halve the waves per SIMD, and measured 0-15% slower.
//
// Measured (a chain of launches in a graph, weights from HBM, us; before =
// proj_mfma_kernel), norm + gate|up + SwiGLU / down + add:
//   8 rows, 2560 x  9728 (100 / 50 MB): 46.3 -> 26.1 / 22.8 -> 13.0
//   8 rows, 4096 x 12288:               60.4 -> 43.5 / 30.3 -> 20.2
//   8 rows, 1024 x  3072:                8.6 ->  7.4 /  4.9 ->  4.9
//  16 rows, 2560 x  9728:               56.9 -> 31.5 / 27.2 -> 15.6
#include <hip/hip_runtime.h>

#include "projection.hpp"

namespace anelm {

namespace {

// Orders the wave's LDS accesses before it before those after it, for lanes
// that hand each other values: a wave's LDS instructions complete in order, so
// this only holds the compiler to the order written (no instruction, no wait;
// 2560 x 9728 at 8 rows takes the same 26.1 / 13.0 us).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Rows, inputs and x rows past the end load the last ones and are not used.
template <int XM, int XR, int NW, int EPI>
__global__ __launch_bounds__(64 * NW) void proj_rows_kernel(ProjArgs a) {
    constexpr bool NORM = XM == kXNorm, X16 = XM == kXF16, PAIR = is_swiglu(EPI);
    constexpr int RT = PAIR ? 2 : 1;              // 16-row tiles of W
    constexpr int ROWS = 4 * XR;                  // rows of x staged
    constexpr int XL = X16 ? XR : 2 * XR;         // x loads per chunk and lane
    __shared__ nat_u32x4 s_w[NW][RT][16][16];     // a wave's chunk of W: row, 8-input piece
    __shared__ nat_u32x4 s_x[NW][ROWS][16];
    __shared__ float s_scale[NORM ? ROWS : 1];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int g = lane >> 4, c = lane & 15;
    const long row0 = (long)blockIdx.x * 16;
    const int K = a.in_dim, nch = (K + 127) / 128;
    // W: load i of a chunk covers rows 4i .. 4i+3, 256 bytes of each; bytes
    // from the tile's first row, the same for gate and up rows
    uint32_t wo[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const long r = row0 + 4 * i + g;
        wo[i] = (uint32_t)((r < a.out_dim ? r : a.out_dim - 1) - row0) * (uint32_t)K * 2u;
    }
    const char* wb0 = reinterpret_cast<const char*>(a.w + row0 * K);
    const char* wb1 = reinterpret_cast<const char*>(a.w + (row0 + a.pair_rows) * K);
    const float* xf = static_cast<const float*>(a.x);
    const char* xb0 = static_cast<const char*>(a.x);
    uint32_t xo[XL];
#pragma unroll
    for (int i = 0; i < XL; i++) {
        const int r = X16 ? 4 * i + g : 2 * i + (lane >> 5);
        xo[i] = (uint32_t)(r < a.batch ? r : a.batch - 1) * (uint32_t)a.ld_x * (X16 ? 2u : 4u);
    }
    nat_u32x4 wr[RT][4], xr[XL];
    uint2 gr;
    auto issue = [&](int q) {
        q = q < nch ? q : nch - 1;
        const int k = min(128 * q + 8 * c, K - 8);
#pragma unroll
        for (int t = 0; t < RT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) wr[t][i] = *reinterpret_cast<const nat_u32x4*>((t == 0 ? wb0 : wb1) + (wo[i] + 2u * (uint32_t)k));
        const int kf = min(128 * q + 4 * (lane & 31), K - 4);
#pragma unroll
        for (int i = 0; i < XL; i++)
            xr[i] = *reinterpret_cast<const nat_u32x4*>(xb0 + (xo[i] + (X16 ? 2u * (uint32_t)k : 4u * (uint32_t)kf)));
        if constexpr (NORM) gr = *reinterpret_cast<const uint2*>(a.gamma + kf);
    };
    constexpr int NPRE = 4;
    float4 pre[NORM ? NPRE : 1];
    auto norm_loads = [&](int r, int k0) {
#pragma unroll
        for (int u = 0; u < NPRE; u++) {
            const int k = k0 + 4 * lane + 256 * u;
            pre[u] = k < K ? *reinterpret_cast<const float4*>(xf + (long)r * a.ld_x + k) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    if constexpr (NORM) {
        if (wv < a.batch) norm_loads(wv, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
    issue(wv);
    float yprev[4];
    if constexpr (EPI == kAdd) {
        const float* y = a.y + (long)(c < a.batch ? c : a.batch - 1) * a.ld_y;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const long r = row0 + 4 * g + i;
            yprev[i] = y[r < a.out_dim ? r : a.out_dim - 1];
        }
    }
    float sc[NORM ? XL : 1];
    if constexpr (NORM) {
        for (int r = wv; r < a.batch; r += NW) {
            float sp[4] = {0.f, 0.f, 0.f, 0.f};
            if (r != wv) norm_loads(r, 0);
            for (int k0 = 0; k0 < K; k0 += 256 * NPRE) {
                if (k0) norm_loads(r, k0);
#pragma unroll
                for (int u = 0; u < NPRE; u++) {
                    sp[u & 3] = fmaf(pre[u].x, pre[u].x, sp[u & 3]);
                    sp[u & 3] = fmaf(pre[u].y, pre[u].y, sp[u & 3]);
                    sp[u & 3] = fmaf(pre[u].z, pre[u].z, sp[u & 3]);
                    sp[u & 3] = fmaf(pre[u].w, pre[u].w, sp[u & 3]);
                }
            }
            const float ss = wave_sum_rows((sp[0] + sp[1]) + (sp[2] + sp[3]));
            if (lane == 0) s_scale[r] = 1.0f / sqrtf(ss / (float)K + a.eps);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < XL; i++) {
            const int r = 2 * i + (lane >> 5);
            sc[i] = s_scale[r < a.batch ? r : a.batch - 1];
        }
    }
    float4v acc[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
    for (int q = wv; q < nch; q += NW) {
#pragma unroll
        for (int t = 0; t < RT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) s_w[wv][t][4 * i + g][c ^ (4 * i + g)] = wr[t][i];
#pragma unroll
        for (int i = 0; i < XL; i++) {
            if constexpr (X16) {
                s_x[wv][4 * i + g][c ^ (4 * i + g)] = xr[i];
            } else {
                const int r = 2 * i + (lane >> 5), p = lane & 31;
                float4 v = __builtin_bit_cast(float4, xr[i]);
                if constexpr (NORM) v = norm_scale(v, sc[i], gr.x, gr.y);
                uint2* dst = reinterpret_cast<uint2*>(&s_x[wv][r][(p >> 1) ^ r]) + (p & 1);
                *dst = make_uint2(pack_f16(v.x, v.y), pack_f16(v.z, v.w));
            }
        }
        if (q + NW < nch) issue(q + NW);   // in flight during this chunk's MFMAs
        wave_lds_sync();
        const int xc = c < ROWS ? c : ROWS - 1;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (128 * q + 32 * s < K) {   // uniform
                const half8 xb = __builtin_bit_cast(half8, s_x[wv][xc][(4 * s + g) ^ xc]);
#pragma unroll
                for (int t = 0; t < RT; t++)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(half8, s_w[wv][t][c][(4 * s + g) ^ c]), xb, acc[t], 0, 0, 0);
            }
        }
        wave_lds_sync();   // the next chunk takes the same places
    }
    // the waves' sums in a fixed order (each wave's go into its own W area)
    float4v* part = reinterpret_cast<float4v*>(&s_w[wv][0][0][0]);
#pragma unroll
    for (int t = 0; t < RT; t++) part[64 * t + lane] = acc[t];
    __syncthreads();
    if (wv > 0 || c >= a.batch) return;
    const float4v* p0 = reinterpret_cast<const float4v*>(&s_w[0][0][0][0]) + lane;
    float4v s = p0[0], u = PAIR ? p0[64] : s;
#pragma unroll
    for (int w = 1; w < NW; w++) {
        s += p0[(long)w * RT * 256];
        if constexpr (PAIR) u += p0[(long)w * RT * 256 + 64];
    }
    const long r = row0 + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (r + i >= a.out_dim) continue;
        const long o = (long)c * a.ld_y + r + i;
        if constexpr (EPI == kAdd) a.y[o] = yprev[i] + r16(s[i]);
        else if constexpr (EPI == kSwiGLU) a.y[o] = silu_ref(r16(s[i])) * r16(u[i]);
        else if constexpr (EPI == kSwiGLU16) a.y16[o] = __builtin_bit_cast(uint16_t, to_f16(silu_ref(r16(s[i])) * r16(u[i])));
        else if constexpr (EPI == kStore16) a.y16[o] = __builtin_bit_cast(uint16_t, to_f16(s[i]));
        else a.y[o] = r16(s[i]);
    }
}

template <int XM, int XR, int NW, int EPI>
void launch_shape(const ProjArgs& a, hipStream_t st) {
    proj_rows_kernel<XM, XR, NW, EPI><<<dim3((unsigned)((a.out_dim + 15) / 16)), dim3(64 * NW), 0, st>>>(a);
}

}  // namespace

bool rows_takes(const ProjArgs& a) {
    return a.batch <= 16 && a.in_dim < (1 << 24) && a.ld_x < (1 << 24);   // 32-bit offsets within a tile and within x
}

// x rows staged: 4, 8 or 16.  Eight waves split a row's chunks, or four from
// 512 workgroups up, which fill the chip by themselves (8 rows: 2560 x 9728
// down, 160 workgroups, 14.0 us with eight and 19.8 with four; gate|up, 608,
// 32.2 and 26.0).  The choice must not depend on the form of x: fp32 rows that
// are fp16 values and the fp16 rows themselves give the same bits.
template <int XM, int EPI>
void launch_rows(const ProjArgs& a, hipStream_t st) {
    const bool wide = a.out_dim >= 16 * 512;
    if (a.batch <= 4) {
        if (wide) launch_shape<XM, 1, 4, EPI>(a, st);
        else launch_shape<XM, 1, 8, EPI>(a, st);
    } else if (a.batch <= 8) {
        if (wide) launch_shape<XM, 2, 4, EPI>(a, st);
        else launch_shape<XM, 2, 8, EPI>(a, st);
    } else {
        if (wide) launch_shape<XM, 4, 4, EPI>(a, st);
        else launch_shape<XM, 4, 8, EPI>(a, st);
    }
}

#define ROWS(XM, EPI) template void launch_rows<XM, EPI>(const ProjArgs&, hipStream_t);
ROWS(kXF32, kStore)
ROWS(kXF32, kAdd)
ROWS(kXF32, kSwiGLU)
ROWS(kXF32, kSwiGLU16)
ROWS(kXNorm, kStore)
ROWS(kXNorm, kAdd)
ROWS(kXNorm, kSwiGLU)
ROWS(kXNorm, kSwiGLU16)
ROWS(kXF16, kStore)
ROWS(kXF16, kAdd)
ROWS(kXF16, kSwiGLU)
ROWS(kXF16, kSwiGLU16)
ROWS(kXF16, kStore16)
#undef ROWS

}  // namespace anelm
