"""The k > 8 top-k block's two ways, by filtering and counting and by sorting, against
oracle.topk_reference (ids and values exact): survivor counts on both sides of the slot counts,
rows whose order or ties defeat the filter, and row lengths at the edges of chunks."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import say

pytestmark = pytest.mark.gpu


def _check(pkg, oracle, lg, k, mode, gpu):
    ids, vals = pkg.logits_topk(torch.from_numpy(lg).to(gpu), k, "sampler" if mode else "f32")
    wi, wv = oracle.topk_reference(lg, k, mode)
    assert np.array_equal(ids.cpu().numpy(), wi)
    assert np.array_equal(vals.cpu().numpy(), wv, equal_nan=True)


@pytest.mark.parametrize("count", [63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 4096])
def test_survivor_counts(gpu, pkg, oracle, count):
    """One block of 4096: `count` logits of 1 or more that touch 64 lane quads (from 64 on),
    the rest 0: where they are equal, exactly those reach the bound."""
    say(f"topk survivors {count}")
    rng = np.random.default_rng(count)
    lead = np.arange(64) * 16 + rng.integers(0, 16, 64)
    rest = rng.permutation(np.setdiff1d(np.arange(4096), lead))
    at = np.concatenate((lead, rest))[:count]
    for ties in (False, True):
        lg = np.zeros((2, 4096), np.float32)
        lg[0, at] = 1.0 if ties else 1.0 + rng.permutation(count).astype(np.float32)
        lg[1, at] = 1.0 if ties else 2.0 + rng.random(count).astype(np.float32)
        for k in (9, 64):
            _check(pkg, oracle, lg, k, 0, gpu)


@pytest.mark.parametrize("n", [9, 64, 65, 1023, 1024, 2048, 4095, 4096, 4097, 8193, 12289, 128256, 270000])
def test_orders_and_lengths(gpu, pkg, oracle, n):
    say(f"topk orders n={n}")
    rng = np.random.default_rng(n)
    up = np.arange(n, dtype=np.float32) - n // 2
    lg = np.stack((up, up[::-1].copy(), np.zeros(n, np.float32), np.full(n, -np.inf, np.float32),
                   np.full(n, np.nan, np.float32), rng.standard_normal(n).astype(np.float32),
                   np.where(rng.random(n) < 0.5, np.nan, rng.standard_normal(n)).astype(np.float32),
                   (up // 64)))
    for k in (9, 40, 64):
        for mode in (0, 1):
            _check(pkg, oracle, lg, k, mode, gpu)
