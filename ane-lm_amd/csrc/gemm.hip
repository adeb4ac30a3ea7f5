// The fp16 projections of projection.hip against many rows of x (a prompt or
// a large batch), where the work is bound by the matrix cores and by how often
// the operands are fetched, no longer by streaming W once.
//
// A workgroup computes 16*TM batch rows x 64*TN outputs with four waves side
// by side along the outputs, each holding TM x TN accumulator tiles of
// v_mfma_f32_16x16x32_f16 (operands and lane layout as in proj_mfma_kernel).
// The x tiles go through LDS, double-buffered and in lane order (1 KB per
// tile, so neither the 16-byte writes nor the reads conflict), because all
// four waves need them; the W tiles are needed by one wave only and go from
// cache straight to its registers, one iteration (KS steps of 32 inputs)
// ahead.  That keeps LDS at TM KB read per 16*TM*TN MFMA cycles and wave, half
// of what staging both operands would take.  With KW > 1, KW such groups of
// waves share the steps of one block, each with its own staging area, and add
// their sums through LDS in a fixed order at the end: few large blocks leave
// each CU bound by the latency of one group's loads, and more waves hide it.
// Workgroups are dealt so that each XCD owns a contiguous run of blocks, batch
// blocks fastest: the blocks in flight on one XCD share a few W tiles in its
// L2, and W leaves HBM about once.  x does not stay there: each column of
// blocks reads all of it again, from the Infinity Cache (gate|up of 2048 rows
// of 4096 x 12288 reads 1.7 GB past the L2 for 218 MB of operands).
//
// Measured with x and W tiled (gate|up + SwiGLU / down + add, us; before =
// proj_mfma_kernel, which fetched W again for every 32 or 64 batch rows):
//   2048 rows, 4096 x 12288: 1541 -> 405 (1018 TFLOP/s) / 1106 -> 198 (1039)
//    500 rows, 2560 x  9728:  209 -> 60 / 132 -> 48
//    100 rows, 4096 x 12288:   92 -> 41 / 68 -> 40
//   1000 rows, 1024 x  3072:   41 -> 20 / 31 -> 20
// (a library GEMM of 8192^3 reaches 1240 TFLOP/s on the same card; inside the
// whole MLP block, x and h fresh from other kernels, 437 and 259 under the
// profiler, 691 in all, with the matrix cores busy 49% and 37% of the time).
// The fp32 sums run in one chain over the inputs with one group, two and four
// with more: of 2048 x 4096 outputs of 12288 inputs 0.32% are not the exact sum
// rounded to fp16, where four chains left 0.25%; the error against 64 bits is
// the rounding's 2.0778e-4 either way.  Blocks of 128 or 256 batch rows
// measured slower throughout (one or two waves per SIMD leave the loads'
// latency bare), as did 2 or 4 steps per iteration for the 64 x 256 block.
#include <hip/hip_runtime.h>

#include "projection.hpp"

namespace anelm {

namespace {

constexpr int kXcds = 8;

// EPI, TILED, XT as in proj_mfma_kernel.  The SwiGLU's waves hold TN/2 gate
// tiles and the TN/2 up tiles pair_rows further on.  Rows, tiles and steps
// past the end load the last one and are not stored (or not computed).
template <int TM, int TN, int KS, int KW, int EPI, bool TILED, bool XT>
__global__ __launch_bounds__(256 * KW) void proj_gemm_kernel(ProjArgs a, int mb, int nb) {
    constexpr bool PAIR = is_swiglu(EPI);
    constexpr int NT = PAIR ? TN / 2 : TN;        // output tiles per wave
    static_assert((TM % 4 == 0 || (4 % TM == 0 && KS * TM % 4 == 0)) && TN % 2 == 0, "tile shape");
    static_assert(KW == 1 || 2 * KS * TM * KW >= 4 * TM * TN, "the partial sums fit the staging area");
    __shared__ nat_u32x4 xs_all[KW][2][KS][TM][64];
    const int lane = threadIdx.x & 63, wv = (threadIdx.x >> 6) & 3, kg = threadIdx.x >> 8;
    auto& xs = xs_all[KW == 1 ? 0 : kg];
    const int g = lane >> 4, c = lane & 15;
    // workgroups go to the XCDs in turn: XCD i takes the i-th run of blocks
    const int total = mb * nb;
    const int xcd = (int)blockIdx.x % kXcds, per = total / kXcds, rem = total % kXcds;
    const int tile = xcd * per + min(xcd, rem) + (int)blockIdx.x / kXcds;
    const int bm = tile % mb, bn = tile / mb;

    const int S = a.in_dim / 32;
    const long ntile = (a.out_dim + 15) / 16;
    const long wstep = TILED ? 512 : 32, xstep = XT ? 512 : 32;
    const uint16_t* wp[TN];
#pragma unroll
    for (int n = 0; n < TN; n++) {
        const bool up = PAIR && n >= NT;
        long t = ((long)bn * 4 + wv) * NT + (up ? n - NT : n);
        if constexpr (TILED) {
            t = t < ntile ? t : ntile - 1;
            if (up) t += a.pair_rows / 16;
            wp[n] = a.w + (t * S * 64 + lane) * 8;
        } else {
            long r = 16 * t + c;
            r = (r < a.out_dim ? r : a.out_dim - 1) + (up ? a.pair_rows : 0);
            wp[n] = a.w + r * a.in_dim + 8 * g;
        }
    }
    // piece j of this wave's staging: piece 4j + wv of the iteration's KS steps x TM tiles
    constexpr int XT4 = TM >= 4 ? TM / 4 : 1;     // x tiles a wave stages
    constexpr int XK = TM >= 4 ? KS : KS * TM / 4; // of so many steps
    const int xt0 = TM >= 4 ? wv : wv % TM, xk0 = TM >= 4 ? 0 : wv / TM;
    constexpr int XKS = TM >= 4 ? 1 : 4 / TM;     // their distance
    const uint16_t* xh = static_cast<const uint16_t*>(a.x);
    const uint16_t* xp[XT4];
#pragma unroll
    for (int j = 0; j < XT4; j++) {
        const long bt = (long)bm * TM + 4 * j + xt0;
        if constexpr (XT) {
            const long last = (a.batch - 1) / 16;
            xp[j] = xh + ((bt < last ? bt : last) * S * 64 + lane) * 8;
        } else {
            const long b = 16 * bt + c;
            xp[j] = xh + (b < a.batch ? b : a.batch - 1) * a.ld_x + 8 * g;
        }
    }

    nat_u32x4 wa[KS][TN], wb[KS][TN], xr[XK][XT4];
    auto load_w = [&](nat_u32x4 (&w)[KS][TN], int it) {
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const int s = min((it * KW + kg) * KS + k, S - 1);
#pragma unroll
            for (int n = 0; n < TN; n++) w[k][n] = *reinterpret_cast<const nat_u32x4*>(wp[n] + s * wstep);
        }
    };
    auto load_x = [&](nat_u32x4 (&xr)[XK][XT4], int it) {
#pragma unroll
        for (int k = 0; k < XK; k++) {
            const int s = min((it * KW + kg) * KS + k * XKS + xk0, S - 1);
#pragma unroll
            for (int j = 0; j < XT4; j++) xr[k][j] = *reinterpret_cast<const nat_u32x4*>(xp[j] + s * xstep);
        }
    };
    auto store_x = [&](const nat_u32x4 (&xr)[XK][XT4], int buf) {
#pragma unroll
        for (int k = 0; k < XK; k++)
#pragma unroll
            for (int j = 0; j < XT4; j++) xs[buf][k * XKS + xk0][4 * j + xt0][lane] = xr[k][j];
    };
    float4v acc[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; m++)
#pragma unroll
        for (int n = 0; n < TN; n++) acc[m][n] = float4v{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const nat_u32x4 (&w)[KS][TN], int buf, int it) {
#pragma unroll
        for (int k = 0; k < KS; k++) {
            if ((it * KW + kg) * KS + k < S) {   // uniform
#pragma unroll
                for (int m = 0; m < TM; m++) {
                    const half8 xb = __builtin_bit_cast(half8, xs[buf][k][m][lane]);
#pragma unroll
                    for (int n = 0; n < TN; n++)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, w[k][n]), xb, acc[m][n], 0, 0, 0);
                }
            }
        }
    };
    const int iters = (S + KS * KW - 1) / (KS * KW);
    load_x(xr, 0);
    load_w(wa, 0);
    store_x(xr, 0);
    load_x(xr, 1);
    __syncthreads();
    for (int it = 0; it < iters; it += 2) {
        load_w(wb, it + 1);
        __builtin_amdgcn_sched_barrier(0);
        compute(wa, 0, it);
        store_x(xr, 1);
        load_x(xr, it + 2);
        __syncthreads();
        load_w(wa, it + 2);
        __builtin_amdgcn_sched_barrier(0);
        compute(wb, 1, it + 1);
        store_x(xr, 0);
        load_x(xr, it + 3);
        __syncthreads();
    }

    if constexpr (KW > 1) {
        // the groups' partial sums, added in a fixed order through the staging area
        float4v* part = reinterpret_cast<float4v*>(&xs_all[0][0][0][0][0]) + wv * TM * TN * 64 + lane;
#pragma unroll
        for (int q = 1; q < KW; q++) {
            if (kg == q) {
#pragma unroll
                for (int m = 0; m < TM; m++)
#pragma unroll
                    for (int n = 0; n < TN; n++) part[(m * TN + n) * 64] = acc[m][n];
            }
            __syncthreads();
            if (kg == 0) {
#pragma unroll
                for (int m = 0; m < TM; m++)
#pragma unroll
                    for (int n = 0; n < TN; n++) acc[m][n] += part[(m * TN + n) * 64];
            }
            if (q + 1 < KW) __syncthreads();
        }
        if (kg) return;
    }
    // lane: outputs 16t + 4g + i of batch row 16m + c
#pragma unroll
    for (int m = 0; m < TM; m++) {
        const long b = ((long)bm * TM + m) * 16 + c;
        if (b >= a.batch) continue;
#pragma unroll
        for (int n = 0; n < NT; n++) {
            const long r = (((long)bn * 4 + wv) * NT + n) * 16 + 4 * g;
            float v[4];
            uint16_t h[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (PAIR) v[i] = silu_ref(r16(acc[m][n][i])) * r16(acc[m][n + NT][i]);
                else v[i] = r16(acc[m][n][i]);
                h[i] = __builtin_bit_cast(uint16_t, to_f16(v[i]));
            }
            const uint2 hv = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
            if constexpr (EPI == kSwiGLU16T) {
                if (r < a.out_dim) *reinterpret_cast<uint2*>(a.y16 + tiled_index(b, (int)r, a.out_dim)) = hv;
            } else if constexpr (EPI == kSwiGLU16 || EPI == kStore16) {
                uint16_t* y = a.y16 + b * a.ld_y + r;
                if (a.vec_y && r + 3 < a.out_dim) {
                    *reinterpret_cast<uint2*>(y) = hv;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (r + i < a.out_dim) y[i] = h[i];
                }
            } else {
                float* y = a.y + b * a.ld_y + r;
                if (a.vec_y && r + 3 < a.out_dim) {
                    float4 o = make_float4(v[0], v[1], v[2], v[3]);
                    if constexpr (EPI == kAdd) {
                        const float4 p = *reinterpret_cast<const float4*>(y);
                        o = make_float4(p.x + o.x, p.y + o.y, p.z + o.z, p.w + o.w);
                    }
                    *reinterpret_cast<float4*>(y) = o;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (r + i < a.out_dim) y[i] = EPI == kAdd ? y[i] + v[i] : v[i];
                }
            }
        }
    }
}

template <int TM, int TN, int KS, int KW, int EPI, bool TILED, bool XT>
void launch_shape(const ProjArgs& a, hipStream_t st) {
    const int bn = 64 * (is_swiglu(EPI) ? TN / 2 : TN);
    const int mb = (a.batch + 16 * TM - 1) / (16 * TM), nb = (a.out_dim + bn - 1) / bn;
    proj_gemm_kernel<TM, TN, KS, KW, EPI, TILED, XT><<<dim3((unsigned)mb * nb), dim3(256 * KW), 0, st>>>(a, mb, nb);
}

// The block shape, 0 where the kernels for few rows stay: 1 = 32 x 128 in two
// groups, 2 = 64 x 128 in four, 3 = 64 x 128 in one, 4 = 64 x 256 in one.  The
// lines were measured over 17-2048 rows at five hidden x intermediate sizes,
// 896 x 4864 to 4096 x 12288, both projections of the MLP, x and W tiled or
// row-major (the shape must not depend on the layout: the outputs of the
// layouts are bit-identical).  nb32, nb64: blocks of 32 or 64 rows by 128
// outputs.
//   - Up to 128 small blocks the other kernel's 16 or 32 row tiles are at most
//     a workgroup per CU, here half the CUs idle and each pulls W through one
//     CU's port: 64 rows of 1024 x 3072 down 8.1 us against 13.0; 500 rows of
//     1024 x 3072 gate|up, 128 blocks, row-major 22.9 against 30.5, tiled 11 to
//     33% slower at 4096 inputs.  Past 128 it loses nowhere in a sweep of 48
//     to 1000 rows, 512 to 9728 inputs, each layout and epilogue (130 to 144
//     blocks: 0.41 to 0.99 of its time).  Long sums without a SwiGLU win from
//     128 on: 100 rows of 4096 x 12288 down 67 -> 64 tiled, 131 -> 116.
//   - Up to one small block per CU nothing else fills the chip (140 rows of
//     1024 x 3072 gate|up: 7.7 us, 64 x 128 blocks 9.5).
//   - 64 x 128 in four groups up to one block per CU (2048 rows of 1024 x 3072
//     down: 23.3 us, one group 26.3, small blocks 28.4), and for long sums up
//     to two (800 rows of 4096 x 12288 down: 116, one group 134); sums under
//     1024 inputs are too short to split in four (200 rows of 896 x 4864
//     gate|up: 16.0, one group 12.2).
//   - 64 x 256 once there are enough blocks for three per CU (500 rows of 2560
//     x 9728 gate|up, 1216 blocks of 64 x 128: 60 against 64), 64 x 128 below
//     (140 rows of 4096 x 12288 gate|up, 576: 54 against 56).
int gemm_shape(const ProjArgs& a, int epi) {
    const long cols = is_swiglu(epi) ? 2L * a.out_dim : a.out_dim;
    const long n128 = (cols + 127) / 128, K = a.in_dim;
    const long nb32 = (a.batch + 31) / 32 * n128, nb64 = (a.batch + 63) / 64 * n128;
    if (a.batch <= 16 || nb32 < (K >= 8192 && !is_swiglu(epi) ? 128 : 129)) return 0;
    if (nb32 > (1L << 30)) return 0;   // the launch's block count is an int
    if (nb32 <= 256) return 1;
    if (nb64 <= 256) return K >= 1024 ? 2 : 3;
    if (nb32 <= 512) return 1;
    if (K >= 4096) return nb64 <= 512 ? 2 : 4;
    return nb64 < 700 ? 3 : 4;
}

}  // namespace

bool gemm_takes(const ProjArgs& a, int epi) { return gemm_shape(a, epi) != 0; }

template <int EPI, bool TILED, bool XT>
void launch_gemm(ProjArgs a, hipStream_t st) {
    constexpr bool f16 = EPI == kSwiGLU16 || EPI == kStore16;
    a.vec_y = f16 ? aligned8(a.y16) && a.ld_y % 4 == 0 : aligned16(a.y) && a.ld_y % 4 == 0;
    switch (gemm_shape(a, EPI)) {
        case 1: launch_shape<2, 2, 2, 2, EPI, TILED, XT>(a, st); break;
        case 2: launch_shape<4, 2, 1, 4, EPI, TILED, XT>(a, st); break;
        case 3: launch_shape<4, 2, 2, 1, EPI, TILED, XT>(a, st); break;
        default: launch_shape<4, 4, 1, 1, EPI, TILED, XT>(a, st); break;
    }
}

#define GEMM(EPI)                                                  \
    template void launch_gemm<EPI, false, false>(ProjArgs, hipStream_t); \
    template void launch_gemm<EPI, true, false>(ProjArgs, hipStream_t);  \
    template void launch_gemm<EPI, true, true>(ProjArgs, hipStream_t);
GEMM(kStore)
GEMM(kAdd)
GEMM(kSwiGLU)
GEMM(kSwiGLU16)
GEMM(kStore16)
template void launch_gemm<kSwiGLU16T, true, true>(ProjArgs, hipStream_t);
#undef GEMM

}  // namespace anelm
