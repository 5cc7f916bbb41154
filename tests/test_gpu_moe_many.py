"""The routed MoE block with many pairs per expert (chunks of 32 pairs, two 16-token blocks per
weight tile): a token's output must be bit for bit what the same token gives in a small batch,
where the one- and four-accumulator kernels run; those are held to the oracle elsewhere."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import say

pytestmark = pytest.mark.gpu


def _experts(pkg, oracle, gpu, E, H, F, rng):
    def pack(n, k):
        return pkg.pack_q4_1(oracle.baseline_q4_1_blocks(n, k, rng), gpu)
    return (pkg.PackedExperts(pack(E * 2 * F, H).data, E, 2 * F, H), pkg.PackedExperts(pack(E * H, F).data, E, H, F))


# per-expert pair counts around the block (16) and chunk (32) edges, an unused expert, ids outside
# [0, E); H of whole and odd 128-row spans (two or one row groups per down workgroup)
@pytest.mark.parametrize("H,F", [(256, 128), (192, 64)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts", [[32, 33, 0, 64, 65, 31], [1, 8, 9, 16, 17, 200], [100, 0, 0, 0, 0, 0]])
def test_many_pairs_equal_small_batches(gpu, pkg, oracle, H, F, xdt, counts):
    say(f"moe many H={H} F={F} {xdt} {counts}")
    E, topk = len(counts), 1
    rng = np.random.default_rng(H + sum(counts))
    gu, dn = _experts(pkg, oracle, gpu, E, H, F, rng)
    ids = np.concatenate([np.full(c, e) for e, c in enumerate(counts)] + [[-1, E, 1 << 20]])
    rng.shuffle(ids)
    T = len(ids)
    assert T > 12 * E
    ids = torch.from_numpy(ids.astype(np.int32)).view(T, topk).to(gpu)
    w = torch.rand(T, topk, generator=torch.Generator(gpu).manual_seed(1), device=gpu)
    x = torch.randn(T, H, generator=torch.Generator(gpu).manual_seed(2), device=gpu).to(xdt)
    out = pkg.moe_batch(gu, dn, x, ids, w, path="decode")
    step = 2 * E
    for t in range(0, T, step):
        ref = pkg.moe_batch(gu, dn, x[t:t + step], ids[t:t + step], w[t:t + step], path="decode")
        assert torch.equal(out[t:t + step], ref), f"tokens {t}.. differ from a small batch"


# more experts than a wave's threads count (two per thread), as many as can have many pairs (14 x 292 =
# 4088), and the last counts of the other kernels; some experts empty
@pytest.mark.parametrize("E,T", [(129, 1549), (160, 1921), (161, 2255), (200, 2801), (200, 2800), (292, 4090), (292, 4088)])
def test_many_experts(gpu, pkg, oracle, E, T):
    say(f"moe many E={E} T={T}")
    H, F = 128, 64
    rng = np.random.default_rng(E)
    gu, dn = _experts(pkg, oracle, gpu, E, H, F, rng)
    live = rng.permutation(E)[:E - E // 5]
    live = np.union1d(live, [0, E - 1])
    ids = torch.from_numpy(np.concatenate([live, rng.choice(live, T - len(live))]).astype(np.int32)).view(T, 1).to(gpu)
    w = torch.rand(T, 1, generator=torch.Generator(gpu).manual_seed(1), device=gpu)
    x = torch.randn(T, H, generator=torch.Generator(gpu).manual_seed(2), device=gpu).to(torch.bfloat16)
    out = pkg.moe_batch(gu, dn, x, ids, w, path="decode")
    for t in range(0, T, 2 * E):
        assert torch.equal(out[t:t + 2 * E], pkg.moe_batch(gu, dn, x[t:t + 2 * E], ids[t:t + 2 * E], w[t:t + 2 * E], path="decode"))


@pytest.mark.parametrize("T", [33, 64, 97])
def test_many_pairs_with_shared_expert(gpu, pkg, oracle, T):
    say(f"moe many shared T={T}")
    E, H, F, Fs, topk = 4, 256, 128, 192, 2
    rng = np.random.default_rng(T)
    gu, dn = _experts(pkg, oracle, gpu, E, H, F, rng)
    g, u = (pkg.pack_q4_1(oracle.baseline_q4_1_blocks(Fs, H, rng), gpu) for _ in range(2))
    shared = (pkg.interleave_gate_up(g, u), pkg.pack_q4_1(oracle.baseline_q4_1_blocks(H, Fs, rng), gpu))
    gen = torch.Generator(gpu).manual_seed(T)
    ids = torch.randint(0, E, (T, topk), generator=gen, device=gpu, dtype=torch.int32)
    w = torch.rand(T, topk, generator=gen, device=gpu)
    x = torch.randn(T, H, generator=gen, device=gpu).to(torch.bfloat16)
    res = torch.randn(T, H, generator=gen, device=gpu)
    sgw = (torch.randn(H, generator=gen, device=gpu) / 16).to(torch.bfloat16)
    assert T * topk > 12 * E
    run = lambda a, b: pkg.moe_batch(gu, dn, x[a:b], ids[a:b], w[a:b], residual=res[a:b], shared_expert=shared,
                                     shared_gate_w=sgw)
    out = run(0, T)
    for t in range(0, T, 4):
        assert torch.equal(out[t:t + 4], run(t, min(t + 4, T)))
