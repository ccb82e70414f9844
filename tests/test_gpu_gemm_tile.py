"""The tile GEMM (granite4_gemm_fp8, granite4_gemm_fp8_swiglu and
granite4_prefill_gemm, most calls of 17 rows and more) at the edges of its tiles
and rings.

Operands are small multiples of 1/2, so every partial sum is a multiple of 1/4
below 2^24 / 4 and exact in f32 in any order: outputs are compared with a
float64 product bit for bit, and with the general kernels bit for bit, which
the same product reaches with zero columns appended to K (to an odd count of
128 for FP8, to no multiple of 64 for bf16). The shapes (gemm_tile_shapes.py)
name the tile that each runs, and several have more tiles than workgroups: the
ring then runs on from a tile into the next one, or is filled again (K groups).
"""
import sys

import pytest
import torch

import gemm_tile_shapes as shapes
from pkg import layerops

pytestmark = pytest.mark.gpu
L = None


def setup_module(module):
    global L
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    L = layerops()
    torch.cuda.init()
    L.use_stream()


def operands(M, N, K, pad, fp8):
    """A [M][K + pad] (its last pad columns zero) and W [N][K + pad] as the entry points take
    them, and both in float64."""
    g = torch.Generator(device="cuda")
    g.manual_seed(M * 7 + N * 3 + K)
    a = torch.randint(-4, 5, (M, K + pad), generator=g, device="cuda", dtype=torch.int32).float() / 2
    w = torch.randint(-4, 5, (N, K + pad), generator=g, device="cuda", dtype=torch.int32).float() / 2
    a[:, K:] = 0
    w[:, K:] = 0
    codes = w.to(torch.float8_e4m3fn).view(torch.uint8)
    A = a.to(torch.float8_e4m3fn).view(torch.uint8) if fp8 else a.to(torch.bfloat16)
    return A, codes, a.double(), w.double()


def pitched(M, N, gap, dtype, fill):
    """An [M][N] view of rows N + gap apart, and the whole buffer (every element `fill`)."""
    whole = torch.full((M, N + gap), fill, dtype=dtype, device="cuda")
    return whole[:, :N], whole


@pytest.mark.parametrize("fp8,M,N,K", [(True, *s[:3]) for s in shapes.FP8 + shapes.FP8_OTHER] +
                         [(False, *s[:3]) for s in shapes.BF16 + shapes.BF16_OTHER])
def test_gemm_tile_equals_general_path(fp8, M, N, K):
    print(f"gemm tile {'fp8' if fp8 else 'bf16'} M={M} N={N} K={K}", flush=True)
    pad = 128 if fp8 else 32
    A, W, a, w = operands(M, N, K, pad, fp8)
    Wk = W[:, :K].contiguous()
    y = a @ w.t()
    segs = (N // 4 // 2 * 2, N // 2 // 2 * 2)
    sc = torch.ones(N, dtype=torch.float64, device="cuda")
    sc[segs[0]:] = 0.5
    sc[segs[1]:] = 2.0

    def run(tile, kind, out, **kw):
        Ak, wt = (A[:, :K], Wk) if tile else (A, W)
        if fp8:
            L.gemm_fp8(Ak, 0.5, wt, out_kind=kind, scales=(2.0, 1.0, 4.0), segs=segs, out=out, **kw)
        else:
            L.prefill_gemm(Ak, wt, kind, scales=(1.0, 0.5, 2.0), segs=segs, out=out, **kw)

    res = (torch.arange(M * N, device="cuda").reshape(M, N) % 17 - 8).to(torch.bfloat16)
    for gap in (0, 8 if fp8 else 2):
        for kind, dtype in ((L.GEMM_F32, torch.float32), (L.GEMM_BF16, torch.bfloat16),
                            (L.GEMM_RESIDUAL, torch.bfloat16)):
            got = []
            for tile in (True, False):
                out, whole = pitched(M, N, gap, dtype, 77.0)
                kw = {}
                if kind == L.GEMM_RESIDUAL:
                    out.copy_(res)
                    kw = {"residual": out, "resid_scale": 0.5}
                run(tile, kind, out, **kw)
                torch.cuda.synchronize()
                assert (whole[:, N:] == 77.0).all()
                got.append(out)
            want = y * sc
            if kind == L.GEMM_RESIDUAL:
                want = res.double() + 0.5 * want
            # exact in f32, so one rounding to the output's type
            assert torch.equal(got[0], want.float().to(dtype)), (kind, gap)
            assert torch.equal(got[0], got[1]), (kind, gap)


@pytest.mark.parametrize("M,I,K", [s[:3] for s in shapes.SWIGLU + shapes.SWIGLU_OTHER])
def test_gemm_tile_swiglu_equals_general_path(M, I, K):
    print(f"gemm tile swiglu M={M} I={I} K={K}", flush=True)
    A, W, a, w = operands(M, 2 * I, K, 128, True)
    work = L.fp8_workspace(rows=16)
    got = []
    for Ak, wt in ((A[:, :K], W[:, :K].contiguous()), (A, W)):
        act, codes, scale = L.gemm_fp8_swiglu(Ak, 0.125, wt, 0.25, 0.5, work)
        torch.cuda.synchronize()
        got.append((act, codes, scale))
    y = a @ w.t()
    g, u = y[:, :I] / 32, y[:, I:] / 16
    want = g / (1 + torch.exp(-g)) * u
    # f32 SwiGLU (a few 2^-24 of its value) and one rounding to bf16
    assert ((got[0][0].double() - want).abs() <= want.abs() * 2.0 ** -8 * 1.01 + 1e-30).all()
    for t, o in zip(*got):
        assert torch.equal(t, o)
