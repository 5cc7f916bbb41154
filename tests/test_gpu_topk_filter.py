"""The k > 8 top-k block (filtering on the leading bits of the values, then on whole keys, then
once more on what is left, and counting) against oracle.topk_reference, ids and values exact:
survivor counts on both sides of the slot counts, ties and masks, rows whose order defeats the
first filters, and row lengths at the edges of chunks."""
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


@pytest.mark.parametrize("count", [63, 64, 65, 127, 128, 129, 255, 256, 257, 319, 320, 321, 511, 512, 513, 4096])
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


@pytest.mark.parametrize("n", [1000, 4096, 5000, 128256])
@pytest.mark.parametrize("live", [0, 1, 39, 40, 63, 64, 65, 600])
def test_masked_rows(gpu, pkg, oracle, n, live):
    """A few live logits, the rest one value (-inf, the lowest f32, NaN): all of the rest reach the
    bound on the values, and the ids decide which of them fill the list. Also values that
    differ only below the bits the first bound looks at."""
    say(f"topk masked n={n} live={live}")
    rng = np.random.default_rng(n + live)
    rows = [np.full(n, v, np.float32) for v in (-np.inf, np.finfo(np.float32).min, np.nan, 0.0, 20.0)]
    for r in rows:
        r[rng.permutation(n)[:live]] = rng.standard_normal(min(live, n)).astype(np.float32)
    rows.append(np.float32(20) * (1 + np.float32(2.0 ** -23) * rng.integers(0, 8, n).astype(np.float32)))
    lg = np.stack(rows).astype(np.float32)
    for k in (9, 40, 64):
        for mode in (0, 1):
            _check(pkg, oracle, lg, k, mode, gpu)


@pytest.mark.parametrize("full", [0, 1, 12, 13, 17, 18, 19, 32, 48, 63, 64, 65, 100])
def test_whole_groups_lead(gpu, pkg, oracle, full):
    """`full` of a block's 256 groups (four neighbouring lanes with their four keys each, 1024
    apart) hold 16 large values each and, up to 64, the other groups one middling value: from 18 full
    groups on the bound that 64 groups reach leaves more keys (16 full + 64 - full) than the 320
    that are ranked, up to 1009, and they are filtered a second time. With 40 such blocks the pass over their
    keys too."""
    say(f"topk whole groups {full}")
    rng = np.random.default_rng(full)
    q = rng.permutation(256)
    at = lambda g: (1024 * np.arange(4)[:, None, None] + 4 * g[None, :, None] + np.arange(4)[None, None, :]).reshape(-1)
    big, mid = at(q[:full]), 4 * q[full:max(full, 64)]
    for blocks in (1, 40):
        for ties in (False, True):
            lg = np.zeros((2, 4096 * blocks), np.float32)
            for b in range(blocks):
                lg[0, 4096 * b + big] = 1000.0 if ties else 1000.0 + rng.permutation(big.size).astype(np.float32)
                lg[0, 4096 * b + mid] = 1.0 + (0 if ties else rng.permutation(mid.size).astype(np.float32))
            lg[1] = -(np.arange(4096 * blocks) // 4 % 64)                 # every value 64 times per block
            for k in (9, 64):
                _check(pkg, oracle, lg, k, 0, gpu)
