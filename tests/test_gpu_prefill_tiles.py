"""The pipelined prefill GEMM's tile forms at the edges of their ranges: token counts around the
64-token groups a tile instance covers (1 to 4 groups of a 256-token tile, 1 or 2 of a
128-token tile), row counts that leave part of a tile over, and K of whole stages and ending
inside one (K % 64, K % 128), with and without K splits, plain and SwiGLU. Small grids are
planned in 128 x 128 tiles; FORMS holds shapes that are planned in 256-row tiles, with and without
192-row ones, and test_prefill_plan.py holds the plan to that."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import say

pytestmark = pytest.mark.gpu

TOKENS = [1, 63, 64, 65, 127, 128, 129, 192, 193, 255, 257, 321]

# (rows of the planned tiles: 192 beside 256, K split or not, T, N, K). The kernel follows from
# them: T % 256 in 1 .. 192 the ragged ones (1 to 3 groups of 64), K % 64 the tail ones.
FORMS = [
    (256, False, 751, 11008, 64), (256, True, 193, 5632, 5952), (192, False, 449, 8448, 64), (192, True, 200, 5760, 4416),
    (256, True, 1, 6656, 1664), (256, True, 65, 12032, 2624), (256, False, 600, 13568, 640), (256, True, 129, 5632, 3328),
    (192, True, 1, 4416, 2112), (192, False, 257, 13056, 64), (192, True, 65, 10944, 1792), (192, False, 600, 6720, 64),
    (192, True, 129, 5568, 2880), (192, False, 385, 12672, 64),
    (256, True, 1, 8448, 1568), (256, True, 65, 8320, 3104), (256, False, 600, 13312, 224), (256, True, 129, 5888, 3104),
    (256, False, 751, 11840, 32), (256, True, 193, 8384, 3360),
]


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


@pytest.mark.parametrize("rows,split,T,N,K", FORMS)
def test_256_row_forms_against_fp64(gpu, pkg, oracle, rows, split, T, N, K):
    """As above, in both precisions, for the shapes whose grids are large enough for 256-row tiles; and
    an infinite activation in the last K block reaches its own token only."""
    say(f"prefill form {rows} split={split} T={T} N={N} K={K}")
    lib = pkg.load_library()
    assert lib.q4_prefill_tile_rows(T, N, K, 0) == rows and (lib.q4_prefill_split_count(T, N, K) > 1) == split
    rng = np.random.default_rng(N + K)
    w = pkg.pack_q4_1(oracle.baseline_q4_1_blocks(N, K, rng), gpu)
    wd = pkg.dequant(w)
    x = _x(T, K, gpu, T)
    ref = x.double() @ wd.double().T
    inf = x.clone()
    at = T // 2
    inf[at, K - 1] = float("inf")
    keep = torch.arange(T, device=gpu) != at
    for precision in ("fp16", "bf16"):
        y = pkg.gemm_q4_prefill(w, x, precision=precision)
        err = y.double() - ref
        if precision == "fp16":
            e = float((err.abs().amax(1) / ref.abs().amax(1)).max())       # token by token
            assert e <= 1e-3, e
        else:
            e = float((err.norm(dim=1) / ref.norm(dim=1)).max())
            assert e <= 5e-3, e
        yi = pkg.gemm_q4_prefill(w, inf, precision=precision)
        assert torch.equal(yi[at].nan_to_num(nan=7.0), (wd[:, K - 1] * float("inf")).nan_to_num(nan=7.0))
        assert torch.equal(yi[keep], y[keep])


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("T,N,K", [(130, 6144, 1216), (130, 2048, 736), (100, 256, 448)] +
                         [(20, 256, k) for k in (544, 736, 832, 928, 1120, 1216, 1312, 1504, 1600, 1696, 1888, 1984)] +
                         [(512, 4096, 14336)])
def test_split_reduce_adds_the_planes_in_order(gpu, pkg, oracle, T, N, K, precision):
    """Every split count (2 to 16, and planes past the caches): the planes that
    gemm_q4_prefill_partials leaves, added up in order, are the GEMM's output, and with f32
    activations the second pass is added to the first's."""
    say(f"prefill reduce T={T} N={N} K={K} {precision}")
    w = pkg.pack_q4_1(oracle.baseline_q4_1_blocks(N, K, np.random.default_rng(K)), gpu)
    x = _x(T, K, gpu, 5)
    p = pkg.prefill_prepare(x, precision)
    planes = pkg.gemm_q4_prefill_partials(w, p)
    assert planes.shape[0] == pkg.load_library().q4_prefill_split_count(T, N, K) > 1
    s = planes[0].clone()
    for q in range(1, planes.shape[0]):
        s += planes[q]
    assert torch.equal(pkg.gemm_q4_prefill(w, p), s)
    if precision == "fp16":          # f32 x whose remainder pass is the bf16 x's product times 2^-12, exactly
        both = x.float() + 2.0 ** -12 * x.float()
        ref = both.double() @ pkg.dequant(w).double().T
        y = pkg.gemm_q4_prefill(w, both, precision=precision)
        assert float((y.double() - ref).abs().max() / ref.abs().max()) <= 1e-3


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
