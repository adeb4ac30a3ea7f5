"""The tiled activation path of the decode step past 16 sequences: fp16
rows in the tiled layout of anelm_proj_tile_f16 (16 rows x 32 columns per
contiguous 1 KB piece), written by the RMSNorm, the fused attention and the
SwiGLU, and read by anelm_proj_f16_tt.  Each tiled output, untiled, is
bit-identical to its row-major counterpart, and the tiled projection to the
row-major kernels on the same operands (models/llm/qwen3.cpp:497-528)."""
import numpy as np
import pytest

from helpers import assert_bitexact, bf16, dev, host

pytestmark = pytest.mark.gpu
THETA = 1e6
EPS = 1e-6


def untile(flat, rows, cols):
    """The [rows, cols] matrix of a tiled fp16 buffer (piece l of block (t, s)
    holds row 16t + l%16, columns 32s + 8(l//16) .. +7)."""
    tiles = (rows + 15) // 16
    a = np.asarray(flat).reshape(-1)[:tiles * 16 * cols].reshape(tiles, cols // 32, 4, 16, 8)
    return a.transpose(0, 3, 1, 2, 4).reshape(tiles * 16, cols)[:rows]


def tiled_buf(rows, cols):
    import torch

    return torch.full(((rows + 15) // 16 * 16 * cols,), -1, dtype=torch.int16, device="cuda")


@pytest.mark.parametrize("rows,dim", [(64, 1024), (17, 1024), (33, 4096), (5, 96), (100, 2048), (9, 96), (65, 1024), (130, 4096)])
def test_rmsnorm_f16_tiled(hip, rng, rows, dim):
    import torch

    x = dev((2 * rng.standard_normal((rows, dim))).astype(np.float32))
    w = dev(bf16(1 + 0.1 * rng.standard_normal(dim)).view(np.int16)).view(torch.bfloat16)
    ref = torch.empty(rows, dim, dtype=torch.int16, device="cuda")
    hip.rmsnorm_f16(ref, x, w, eps=EPS)
    out = tiled_buf(rows, dim)
    hip.rmsnorm_f16_tiled(out, x, w, eps=EPS)
    assert_bitexact(untile(host(out), rows, dim), host(ref), "tiled RMSNorm vs rows")


def test_rmsnorm_f16_tiled_rejects(hip):
    import torch

    x = torch.zeros(4, 100, device="cuda")
    w = torch.ones(100, device="cuda").bfloat16()
    with pytest.raises(Exception):
        hip.rmsnorm_f16_tiled(torch.zeros(16 * 128, dtype=torch.int16, device="cuda"), x, w)   # dim % 32


@pytest.mark.parametrize("B,nq,nk,cap", [(64, 16, 8, 64), (20, 32, 8, 300), (17, 8, 8, 40)])
def test_attention_qk_tiled_output(hip, orc, rng, B, nq, nk, cap):
    """The fused attention's tiled fp16 output equals its fp16 rows, over
    rings of random start and length (long rings merged across chunks)."""
    import torch

    D = 128
    qkv = rng.standard_normal((B, (nq + 2 * nk) * D), dtype=np.float32)
    pos = rng.integers(0, 3000, B).astype(np.int32)
    wq = dev(bf16(1 + 0.1 * rng.standard_normal(D)).view(np.int16)).view(torch.bfloat16)
    wk = dev(bf16(1 + 0.1 * rng.standard_normal(D)).view(np.int16)).view(torch.bfloat16)
    c_tab, s_tab = orc.rope_table(2048, D, THETA)
    kc0 = rng.standard_normal((B, cap, nk * D), dtype=np.float32)
    vc0 = rng.standard_normal((B, cap, nk * D), dtype=np.float32)
    rs0 = rng.integers(0, cap, B).astype(np.int32)
    rl0 = rng.integers(0, cap + 1, B).astype(np.int32)
    rl0[0] = cap
    outs = []
    for tiled in (False, True):
        a = dev(qkv)
        kc, vc, rs, rl = dev(kc0), dev(vc0), dev(rs0), dev(rl0)
        hip.kv_ring_advance(rs, rl, cap)
        ws = torch.zeros(max(hip.gqa_workspace_size(B, nq, nk, D, cap), 16), dtype=torch.uint8, device="cuda")
        out = tiled_buf(B, nq * D) if tiled else torch.full((B, nq * D), -1, dtype=torch.int16, device="cuda")
        hip.gqa_attention_qk(out, a[:, :nq * D], a[:, nq * D:(nq + nk) * D], a[:, (nq + nk) * D:], wq, wk, dev(pos),
                             dev(c_tab), dev(s_tab), kc, vc, rs, rl, nq, nk, ws, THETA, EPS, tiled=tiled)
        outs.append(untile(host(out), B, nq * D) if tiled else host(out))
    assert_bitexact(outs[1], outs[0], "tiled attention output vs rows")


@pytest.mark.parametrize("B,out_dim,in_dim", [(64, 4096, 1024), (64, 1024, 2048), (64, 1024, 3072), (17, 1000, 256),
                                               (40, 3072, 1024), (20, 6144, 1024), (64, 16, 4096), (18, 512, 1024)])
def test_proj_f16_tt(hip, orc, rng, B, out_dim, in_dim):
    """Tiled x and tiled W: every epilogue bit-identical to the tiled-W
    projection on row-major x; the tiled fp16 SwiGLU, untiled, equals the
    fp16 SwiGLU rows."""
    import torch

    x16 = orc.f32_to_f16_rne((2 * rng.standard_normal((B, in_dim))).astype(np.float32)).reshape(B, in_dim)
    xr = dev(x16.view(np.int16))
    xt = tiled_buf(B, in_dim)
    hip.proj_tile_f16(xt, xr)       # the tiled layout of the rows (the W tiling routine, rows = batch rows)
    assert_bitexact(untile(host(xt), B, in_dim), x16.view(np.int16), "tiled x")
    w = dev((0.03 * rng.standard_normal((out_dim, in_dim))).astype(np.float16).view(np.int16))
    wt = torch.full((hip.proj_tiled_size(out_dim, in_dim) // 2,), -1, dtype=torch.int16, device="cuda")
    hip.proj_tile_f16(wt, w)
    r0 = rng.standard_normal((B, out_dim)).astype(np.float32)
    for epi in (hip.PROJ_STORE, hip.PROJ_ADD):
        y, yr = dev(r0), dev(r0)
        hip.proj_f16_tt(y, xt, wt, B, out_dim, in_dim, epilogue=epi)
        hip.proj_f16_x16_tiled(yr, xr, wt, out_dim, epilogue=epi)
        assert_bitexact(host(y), host(yr), f"tiled x vs rows, epilogue {epi}")
    y16 = torch.empty(B, out_dim, dtype=torch.int16, device="cuda")
    yr16 = torch.empty(B, out_dim, dtype=torch.int16, device="cuda")
    hip.proj_f16_tt(y16, xt, wt, B, out_dim, in_dim, epilogue=hip.PROJ_STORE_F16)
    hip.proj_f16_x16_tiled(yr16, xr, wt, out_dim, epilogue=hip.PROJ_STORE_F16)
    assert_bitexact(host(y16), host(yr16), "tiled x vs rows, fp16 store")
    if out_dim % 32 == 0:
        inter = out_dim // 2
        for epi, dt in ((hip.PROJ_SWIGLU, torch.float32), (hip.PROJ_SWIGLU_F16, torch.int16)):
            h = torch.full((B, inter), -1, dtype=dt, device="cuda")
            hr = torch.full((B, inter), -1, dtype=dt, device="cuda")
            hip.proj_f16_tt(h, xt, wt, B, inter, in_dim, epilogue=epi)
            hip.proj_f16_x16_tiled(hr, xr, wt, inter, epilogue=epi)
            assert_bitexact(host(h), host(hr), f"tiled x vs rows, SwiGLU epilogue {epi}")
        if inter % 32 == 0:
            ht = tiled_buf(B, inter)
            hip.proj_f16_tt(ht, xt, wt, B, inter, in_dim, epilogue=hip.PROJ_SWIGLU_F16_TILED)
            assert_bitexact(untile(host(ht), B, inter), host(hr), "tiled fp16 SwiGLU vs rows")


def test_proj_f16_tt_adjacent_buffers(hip, rng):
    """y's 17 rows followed directly by x_t (32 padded rows) in one buffer:
    accepted (the overlap check takes y's own rows, not x_t's padded count),
    and the result equals the same call on separate buffers."""
    import torch

    B, out_dim, in_dim = 17, 64, 256
    buf = torch.zeros(B * out_dim + 32 * in_dim // 2, dtype=torch.float32, device="cuda")
    y = buf[:B * out_dim].view(B, out_dim)
    xt = buf[B * out_dim:].view(torch.int16)
    x16 = (rng.standard_normal((B, in_dim)) * 0.5).astype(np.float16)
    xr = dev(x16.view(np.int16))
    hip.proj_tile_f16(xt, xr)
    w = dev((0.03 * rng.standard_normal((out_dim, in_dim))).astype(np.float16).view(np.int16))
    wt = torch.zeros(hip.proj_tiled_size(out_dim, in_dim) // 2, dtype=torch.int16, device="cuda")
    hip.proj_tile_f16(wt, w)
    hip.proj_f16_tt(y, xt, wt, B, out_dim, in_dim, epilogue=hip.PROJ_STORE)
    ref = torch.zeros(B, out_dim, device="cuda")
    xt2 = tiled_buf(B, in_dim)
    hip.proj_tile_f16(xt2, xr)
    hip.proj_f16_tt(ref, xt2, wt, B, out_dim, in_dim, epilogue=hip.PROJ_STORE)
    assert_bitexact(host(y), host(ref), "adjacent y and x_t")


# Many rows of x: the block-tiled kernel's four block shapes (chosen by the
# number of blocks), each with a last batch block, output block and input step
# that are only partly there: 1 (129 blocks of 32 x 128; an output count that
# is no multiple of 4, one input step), 1 again (three input steps for two
# groups of two, and 33: nine passes of the double-buffered loop), 2 (256 blocks
# of 64 x 128, 33 steps for four groups), 3 (320 blocks, odd steps), 4 (715
# blocks; two steps, and 33); 4096 or more inputs, where 2 stays up to 512 blocks
# and 4 follows (260 and 585, 129 steps); and fewer blocks than it takes: 24,
# and 128, which it takes from 8192 inputs.
@pytest.mark.parametrize("B,out_dim,in_dim", [(65, 5501, 32), (65, 5504, 96), (17, 16352, 64), (200, 8160, 1056),
                                               (300, 8160, 160), (700, 8288, 64), (70, 1024, 96),
                                               (65, 5504, 1056), (700, 8288, 1056), (256, 8320, 4128), (520, 8320, 4128),
                                               (100, 4096, 96), (100, 4084, 8192)])
def test_many_rows(hip, orc, rng, B, out_dim, in_dim):
    """Every epilogue and layout: within an fp16 ulp of the oracle, tiled
    layouts bit-identical to row-major, fp16 stores the fp32 ones narrowed."""
    import torch
    from test_gpu_qwen3 import _proj_ref, _ulp16, check_projection

    x = (2 * rng.standard_normal((B, in_dim))).astype(np.float32)
    x16 = orc.f32_to_f16_rne(x).reshape(B, in_dim)
    w = (0.03 * rng.standard_normal((out_dim, in_dim))).astype(np.float16).view(np.uint16)
    xr, dw = dev(x16.view(np.int16)), dev(w.view(np.int16))
    xt, wt = tiled_buf(B, in_dim), tiled_buf(out_dim, in_dim)
    hip.proj_tile_f16(xt, xr)
    hip.proj_tile_f16(wt, dw)

    def three(n, epi, dt, y0=None):
        """The output of the row-major call, checked against the two tiled ones."""
        ys = [dev(y0) if y0 is not None else torch.full((B, n), -1, dtype=dt, device="cuda") for _ in range(3)]
        if epi != hip.PROJ_STORE_F16:
            hip.proj_f16_x16_fused(ys[0], xr, dw, epilogue=epi)
        else:
            hip.linear_f16(ys[0], xr, dw)
        hip.proj_f16_x16_tiled(ys[1], xr, wt, n, epilogue=epi)
        hip.proj_f16_tt(ys[2], xt, wt, B, n, in_dim, epilogue=epi)
        for y in ys[1:]:
            assert_bitexact(host(y), host(ys[0]), f"layouts, epilogue {epi}")
        return host(ys[0])

    y = three(out_dim, hip.PROJ_STORE, torch.float32)
    check_projection(orc, x, w, y.astype(np.float64))
    y2 = torch.full((B, out_dim), -1.0, device="cuda")
    hip.proj_f16_x16(y2, xr, dw)
    assert_bitexact(host(y2), y, "proj_f16_x16")
    y16 = three(out_dim, hip.PROJ_STORE_F16, torch.int16)
    assert_bitexact(y16, orc.f32_to_f16_rne(y).reshape(B, out_dim).view(np.int16), "fp16 store")
    r0 = rng.standard_normal((B, out_dim)).astype(np.float32)
    assert_bitexact(three(out_dim, hip.PROJ_ADD, torch.float32, r0), r0 + y, "residual add")
    # one float off a 16-byte boundary: the element-wise stores
    off = torch.full((B * out_dim + 1,), -1.0, device="cuda")
    hip.proj_f16_x16_fused(off[1:].view(B, out_dim), xr, dw)
    assert_bitexact(host(off[1:].view(B, out_dim)), y, "unaligned output")
    if out_dim % 32 == 0:
        n = out_dim // 2
        h = three(n, hip.PROJ_SWIGLU, torch.float32)
        g, u = y[:, :n].astype(np.float64), y[:, n:].astype(np.float64)
        want = g / (1 + np.exp(-g)) * u
        assert np.all(np.abs(h - want) <= 1e-5 * np.abs(want) + 1e-30)
        h16 = three(n, hip.PROJ_SWIGLU_F16, torch.int16)
        assert_bitexact(h16, orc.f32_to_f16_rne(h).reshape(B, n).view(np.int16), "fp16 SwiGLU")
        if n % 32 == 0:
            ht = tiled_buf(B, n)
            hip.proj_f16_tt(ht, xt, wt, B, n, in_dim, epilogue=hip.PROJ_SWIGLU_F16_TILED)
            assert_bitexact(untile(host(ht), B, n), h16, "tiled fp16 SwiGLU")
            pad = np.asarray(host(ht)).reshape((B + 15) // 16, n // 32, 4, 16, 8)[-1, :, :, (B - 1) % 16 + 1:]
            assert np.all(pad.astype(np.uint16) == 0xFFFF), "rows past the batch are left as they are"


# Stores of 8192 or more outputs, all of x in LDS: 64, 32 and 16 rows a
# workgroup, with rows and outputs that are only partly there; and just past the
# rows it holds, where the block-tiled kernel takes over in every layout (and
# proj_mfma_kernel at 128 blocks).
@pytest.mark.parametrize("B,out_dim,in_dim,gemm", [(17, 8192, 256, 0), (64, 8200, 1024, 0), (30, 8208, 2048, 0),
                                                    (20, 8196, 4096, 0), (65, 8192, 1024, 1), (33, 16384, 4096, 1),
                                                    (33, 8192, 2048, 1)])
def test_stores_through_lds(hip, orc, rng, B, out_dim, in_dim, gemm):
    """Every layout with x in rows gives the same bits here too, in fp32 and
    fp16; x tiled takes the kernels that split the inputs over waves, whose sums
    run in another order: its fp16 stores are its fp32 ones, each checked."""
    import torch
    from test_gpu_qwen3 import check_projection

    x = (2 * rng.standard_normal((B, in_dim))).astype(np.float32)
    x16 = orc.f32_to_f16_rne(x).reshape(B, in_dim)
    w = (0.03 * rng.standard_normal((out_dim, in_dim))).astype(np.float16).view(np.uint16)
    xr, dw = dev(x16.view(np.int16)), dev(w.view(np.int16))
    xt, wt = tiled_buf(B, in_dim), tiled_buf(out_dim, in_dim)
    hip.proj_tile_f16(xt, xr)
    # the rows past the batch are padding, whatever they hold
    pad = xt.view((B + 15) // 16, in_dim // 32, 4, 16, 8)[-1, :, :, (B - 1) % 16 + 1:]
    pad.fill_(0x7E00)
    hip.proj_tile_f16(wt, dw)
    out = lambda dt: torch.full((B, out_dim), -1, dtype=dt, device="cuda")  # noqa: E731
    y = [out(torch.float32) for _ in range(4)]
    hip.proj_f16_x16_fused(y[0], xr, dw)
    hip.proj_f16_x16(y[1], xr, dw)
    hip.proj_f16_x16_tiled(y[2], xr, wt, out_dim)
    hip.proj_f16_tt(y[3], xt, wt, B, out_dim, in_dim, epilogue=hip.PROJ_STORE)
    check_projection(orc, x, w, host(y[0]).astype(np.float64))
    check_projection(orc, x, w, host(y[3]).astype(np.float64))
    for i in (1, 2, 3) if gemm else (1, 2):
        assert_bitexact(host(y[i]), host(y[0]), f"layout {i}")
    h = [out(torch.int16) for _ in range(3)]
    hip.linear_f16(h[0], xr, dw)
    hip.proj_f16_x16_tiled(h[1], xr, wt, out_dim, epilogue=hip.PROJ_STORE_F16)
    hip.proj_f16_tt(h[2], xt, wt, B, out_dim, in_dim, epilogue=hip.PROJ_STORE_F16)
    for i, of in enumerate((y[0], y[0], y[3])):
        assert_bitexact(host(h[i]), orc.f32_to_f16_rne(host(of)).reshape(B, out_dim).view(np.int16), f"fp16 store {i}")
