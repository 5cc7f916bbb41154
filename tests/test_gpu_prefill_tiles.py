"""The pipelined prefill GEMM's tile forms at the edges of their ranges: token counts around the
64-token groups a tile instance covers (1 to 4 groups of a 256-token tile, 1 or 2 of a
128-token tile), row counts that leave part of a 256- or 128-row tile over, and K of whole stages
and ending inside one (K % 64, K % 128), with and without K splits, plain and SwiGLU."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import say

pytestmark = pytest.mark.gpu

TOKENS = [1, 63, 64, 65, 127, 128, 129, 192, 193, 255, 257, 321]


def _x(T, K, gpu, seed):
    return torch.randn(T, K, generator=torch.Generator(gpu).manual_seed(seed), device=gpu).to(torch.bfloat16)


@pytest.mark.parametrize("precision,bar", [("fp16", 1e-3), ("bf16", 5e-3)])
@pytest.mark.parametrize("N,K", [(64, 128), (192, 1088), (320, 1152), (4096, 128), (64, 32), (192, 1120), (320, 96),
                                 (4096, 160)])
def test_tiles_against_fp64(gpu, pkg, oracle, N, K, precision, bar):
    """Every token count against fp64 on the dequantized weights, at the library's bars (max-rel
    1e-3; the bf16 tile 5e-3 in the Frobenius norm), and without a K split token rows independent
    of T (either form adds K in the same order)."""
    say(f"prefill tiles N={N} K={K} {precision}")
    blocks = oracle.baseline_q4_1_blocks(N, K, np.random.default_rng(N + K))
    w = pkg.pack_q4_1(blocks, gpu)
    wd = pkg.dequant(w).double()
    x = _x(max(TOKENS), K, gpu, 7)
    lib = pkg.load_library()
    first = None
    for T in TOKENS:
        y = pkg.gemm_q4_prefill(w, x[:T], precision=precision)
        ref = x[:T].double() @ wd.T
        err = (y.double() - ref)
        e = float(err.abs().max() / ref.abs().max()) if precision == "fp16" else float(err.norm() / ref.norm())
        assert e <= bar, f"T={T}: {e:.2e}"
        if lib.q4_prefill_split_count(T, N, K) == 1:
            first = y[:1].clone() if first is None else first
            assert torch.equal(first, y[:1]), f"T={T}: token 0 differs from the other token counts'"


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("F,K", [(128, 128), (128, 192), (384, 1152)])
def test_swiglu_tiles_equal_the_plain_gemm(gpu, pkg, oracle, F, K, precision):
    """The SwiGLU epilogue's h, in either tile form, is bf16(silu(g) u) of the plain GEMM's f32
    gate and up outputs where that GEMM is unsplit (the same bits), else within one bf16
    rounding (2^-8) plus the sums' reordering."""
    say(f"swiglu tiles F={F} K={K} {precision}")
    rng = np.random.default_rng(F + K)
    g, u = (pkg.pack_q4_1(oracle.baseline_q4_1_blocks(F, K, rng), gpu) for _ in range(2))
    gu = pkg.interleave_gate_up(g, u)
    x = _x(max(TOKENS), K, gpu, 9)
    lib = pkg.load_library()
    for T in TOKENS:
        p = pkg.prefill_prepare(x[:T], precision)
        h = pkg.gemm_q4_prefill_swiglu(gu, p)
        ref = torch.empty_like(h)
        pkg.swiglu_prepare(pkg.gemm_q4_prefill(g, p), pkg.gemm_q4_prefill(u, p), precision=precision, h=ref)
        if lib.q4_prefill_split_count(T, F, K) == 1:
            assert torch.equal(h, ref), f"T={T}"
        else:
            d = (h.double() - ref.double()).abs()
            assert float((d - 2.0 ** -7 * ref.double().abs()).max()) <= 1e-6, f"T={T}"


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("T", [5, 300])
@pytest.mark.parametrize("K", [32, 160, 192, 1120, 1088])
def test_tail_planes_leave_infinities_alone(gpu, pkg, oracle, K, T, precision):
    """A K that ends inside a stage: the stage's zeros must meet no data. An infinite activation in
    the last K block gives its token the signed infinities of that column's weights (a NaN for a
    zero weight), and no other token changes."""
    say(f"prefill tail inf K={K} T={T} {precision}")
    N = 192
    w = pkg.pack_q4_1(oracle.baseline_q4_1_blocks(N, K, np.random.default_rng(K)), gpu)
    wd = pkg.dequant(w)
    x = _x(T, K, gpu, 3)
    clean = pkg.gemm_q4_prefill(w, x, precision=precision)
    x[2, K - 1] = float("inf")
    y = pkg.gemm_q4_prefill(w, x, precision=precision)
    want = wd[:, K - 1] * float("inf")
    assert torch.equal(y[2].nan_to_num(nan=7.0), want.nan_to_num(nan=7.0))
    keep = [t for t in range(T) if t != 2]
    assert torch.equal(y[keep], clean[keep])
