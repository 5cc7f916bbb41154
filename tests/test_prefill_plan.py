"""The prefill GEMM's plan, asked on the host (no GPU: the plan then takes the MI355X's 256 CUs):
the shapes that the GPU tests rely on for a tile form are planned in that form, and the split
counts that the reduce has instances for are all met."""
from __future__ import annotations

import pytest

from test_gpu_prefill_tiles import FORMS


@pytest.mark.parametrize("rows,split,T,N,K", FORMS)
def test_forms(lib, rows, split, T, N, K):
    assert lib.q4_prefill_tile_rows(T, N, K, 0) == rows
    assert (lib.q4_prefill_split_count(T, N, K) > 1) == split


@pytest.mark.parametrize("mixed", [False, True])
def test_forms_hold_every_ragged_instance(mixed):
    """1 to 3 groups of 64 tokens in the last tile of a ragged launch, and full ones, for 256-row
    tiles with and without 192-row ones and for K that ends inside a stage."""
    want = {(g, False) for g in (1, 2, 3, 4)} | (set() if mixed else {(g, True) for g in (1, 2, 3, 4)})
    assert {((T - 1) % 256 // 64 + 1, K % 64 != 0) for rows, _, T, _, K in FORMS if (rows == 192) == mixed} == want


def test_split_counts_and_small_grids(lib):
    counts = {lib.q4_prefill_split_count(20, 256, k) for k in range(256, 2048, 32)}
    counts |= {lib.q4_prefill_split_count(T, N, K) for T, N, K in ((130, 6144, 1216), (130, 2048, 736), (100, 256, 448))}
    assert counts >= set(range(1, 17))
    for T in (1, 64, 100, 321):
        assert lib.q4_prefill_tile_rows(T, 192, 1088, 0) == 128
    # SwiGLU: K of odd 64s takes 256-row tiles, whole 128s on a small grid 128-row ones
    assert lib.q4_prefill_tile_rows(321, 256, 192, 1) == 256 and lib.q4_prefill_tile_rows(321, 768, 1152, 1) == 128
