"""Projections of 3 to 16 rows against a row-major W: 16 outputs per workgroup,
128-input chunks dealt to 8 waves (4 from 8192 outputs), 4, 8 or 16 rows of x
staged per wave (core/ane_runtime.cpp:265-408 with ane_matvec :600-640)."""
import numpy as np
import pytest

from helpers import assert_bitexact, bf16, dev, from_bf16, host
from test_gpu_qwen3 import _proj_ref, _ulp16, check_projection

pytestmark = pytest.mark.gpu


# Edges: fewer chunks than waves and a chunk of one step (32, 96 inputs), a
# last chunk that is partly there, more chunks than waves; fewer than 16
# outputs, a ragged last tile, both wave counts (8192 outputs either side); the
# smallest and largest row counts of each staging size; two rows where the dot
# kernel hands over; and where it keeps two to four rows of whole rounds of its
# loads, or with a norm.
@pytest.mark.parametrize("B,out_dim,in_dim", [(3, 10, 32), (4, 8208, 160), (5, 33, 96), (8, 1040, 4128), (9, 16, 1056),
                                               (16, 8191, 64), (6, 8192, 256), (13, 2048, 2080), (2, 2576, 4096),
                                               (2, 3080, 6144), (4, 520, 6144), (3, 1024, 4096)])
def test_few_rows(hip, orc, rng, B, out_dim, in_dim):
    import torch

    x16 = orc.f32_to_f16_rne((2 * rng.standard_normal((B, in_dim))).astype(np.float32)).reshape(B, in_dim)
    x = x16.view(np.float16).astype(np.float32)
    w = (0.03 * rng.standard_normal((out_dim, in_dim))).astype(np.float16).view(np.uint16)
    gamma = bf16(1 + 0.1 * rng.standard_normal(in_dim))
    # rows of a wider buffer, the rest NaN: nothing outside the rows is used
    xw = torch.full((B, in_dim + 8), float("nan"), device="cuda")
    xw[:, :in_dim] = dev(x)
    hw = xw.half()
    xf, xh, dw = xw[:, :in_dim], hw[:, :in_dim], dev(w.view(np.int16))
    r0 = rng.standard_normal((B, out_dim)).astype(np.float32)
    ref, mag = _proj_ref(orc, x, w)
    tol = _ulp16(ref) + mag * 2.0 ** -21 * 4
    for epi, base in ((hip.PROJ_STORE, 0.0), (hip.PROJ_ADD, r0.astype(np.float64))):
        ys = []
        for call, a in ((hip.proj_f16_fused, xf), (hip.proj_f16_x16_fused, xh)):
            yw = torch.full((B, out_dim + 4), float("nan"), device="cuda")
            yw[:, :out_dim] = dev(r0)
            call(yw[:, :out_dim], a, dw, epilogue=epi)
            assert torch.isnan(yw[:, out_dim:]).all(), "written past the row"
            ys.append(host(yw[:, :out_dim].contiguous()))
        assert_bitexact(ys[1], ys[0], f"fp16 rows vs fp32 rows, epilogue {epi}")
        want = base + ref
        assert np.all(np.abs(ys[0].astype(np.float64) - want) <= tol + np.spacing(np.abs(want).astype(np.float32)))
        if epi == hip.PROJ_STORE:
            y16 = torch.empty(B, out_dim, dtype=torch.int16, device="cuda")
            hip.linear_f16(y16, xh, dw)
            check_projection(orc, x, w, host(y16).view(np.float16).astype(np.float64))
    xn = np.stack([orc.rmsnorm(x[b], from_bf16(gamma), 1e-6) for b in range(B)])
    y = torch.full((B, out_dim), float("nan"), device="cuda")
    hip.proj_f16_fused(y, xf, dw, norm=dev(gamma.view(np.int16)), eps=1e-6)
    check_projection(orc, xn, w, host(y).astype(np.float64))
    n = out_dim // 2
    for norm, rows in ((None, x), (dev(gamma.view(np.int16)), xn)):
        h = torch.full((B, n), float("nan"), device="cuda")
        h16 = torch.empty(B, n, dtype=torch.int16, device="cuda")
        hip.proj_f16_fused(h, xf, dw[:2 * n], norm=norm, eps=1e-6, epilogue=hip.PROJ_SWIGLU)
        hip.proj_f16_fused(h16, xf, dw[:2 * n], norm=norm, eps=1e-6, epilogue=hip.PROJ_SWIGLU_F16)
        assert_bitexact(host(h16), orc.f32_to_f16_rne(host(h)).reshape(B, n), "fp16 SwiGLU vs fp32 SwiGLU rounded")
        gu, m = _proj_ref(orc, rows, w[:2 * n])
        g, u = gu[:, :n], gu[:, n:]
        eg, eu = (_ulp16(v) + mm * 2.0 ** -21 * 4 for v, mm in ((g, m[:, :n]), (u, m[:, n:])))
        sg = g / (1 + np.exp(-g))
        lim = 1.1 * eg * np.abs(u) + np.abs(sg) * eu + eg * eu + np.abs(sg * u) * 1e-6 + 1e-30   # silu' <= 1.1
        assert np.all(np.abs(host(h).astype(np.float64) - sg * u) <= lim)
        if norm is None:
            hip.proj_f16_x16_fused(h, xh, dw[:2 * n], epilogue=hip.PROJ_SWIGLU)
            assert_bitexact(orc.f32_to_f16_rne(host(h)).reshape(B, n), host(h16), "SwiGLU of fp16 rows vs fp32 rows")


# 7 and 16 rows: the kernel above; 40: proj_mfma_kernel; 100: block tiles.
@pytest.mark.parametrize("B", [7, 16, 40, 100])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_rows_do_not_mix(hip, rng, B, bad):
    """A NaN or an infinity in a row of x, or of W, reaches that row's outputs
    (that column's) and no others: these keep their bits."""
    import torch

    out_dim, in_dim = 4112, 160
    x = rng.standard_normal((B, in_dim)).astype(np.float32)
    w = (0.03 * rng.standard_normal((out_dim, in_dim))).astype(np.float16)
    xb, wb = x.copy(), w.copy()
    rows, cols = [2, B - 1], [0, 2055, 4111]
    xb[rows, [5, in_dim - 1]] = bad
    wb[cols, [0, 33, in_dim - 1]] = bad
    gamma = dev(bf16(np.ones(in_dim, np.float32)).view(np.int16))
    tiled = lambda a: torch.zeros((a.shape[0] + 15) // 16 * 16 * a.shape[1], dtype=torch.int16, device="cuda")  # noqa: E731

    def calls(x, w):
        xf, dw = dev(x), dev(w.view(np.int16))
        xh = xf.half().view(torch.int16)
        wt, xt = tiled(w), tiled(x)
        hip.proj_tile_f16(wt, dw)
        hip.proj_tile_f16(xt, xh)
        ys = [torch.zeros(B, out_dim, device="cuda") for _ in range(5)]
        hip.proj_f16_fused(ys[0], xf, dw)
        hip.proj_f16_fused(ys[1], xf, dw, norm=gamma, eps=1e-6)
        hip.proj_f16_x16_fused(ys[2], xh, dw)
        hip.proj_f16_x16_tiled(ys[3], xh, wt, out_dim)
        hip.proj_f16_tt(ys[4], xt, wt, B, out_dim, in_dim, epilogue=hip.PROJ_STORE)
        return [host(y) for y in ys]

    clean = calls(x, w)
    for i, (y, of_x, of_w) in enumerate(zip(clean, calls(xb, w), calls(x, wb))):
        keep = np.setdiff1d(np.arange(B), rows)
        assert_bitexact(of_x[keep], y[keep], f"call {i}: other rows")
        assert not np.isfinite(of_x[rows]).any(), f"call {i}: rows of the {bad}"
        keep = np.setdiff1d(np.arange(out_dim), cols)
        assert_bitexact(of_w[:, keep], y[:, keep], f"call {i}: other columns")
        assert not np.isfinite(of_w[:, cols]).any(), f"call {i}: columns of the {bad}"
