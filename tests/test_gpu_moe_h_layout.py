"""The bf16 h rows of a prefill expert block on their way into the down GEMM's layout: expert
populations around the 64-slot groups of a tile, F around the four-slots-per-wave limit (1536)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F", [128, 768, 1536, 1664])
@pytest.mark.parametrize("counts", [(1, 63, 64, 65, 127, 129, 192, 193, 255, 256, 257, 0, 320), (4099,)])
def test_h_rows_at_group_edges(gpu, pkg, oracle, F, counts):
    """The second population has more than 16 tiles for its expert: whole tiles are laid out. The
    bound is the block's own on its oracle (bf16 h, fp16 tiles): 1e-3 of the largest output."""
    say(f"moe h layout F={F} counts={counts}")
    H, E = 256, len(counts)
    rng = np.random.default_rng(F + E)
    gates, ups, downs = ([oracle.baseline_q4_1_blocks(n, k, rng) for _ in range(E)]
                         for n, k in ((F, H), (F, H), (H, F)))
    gu, dn = pkg.pack_moe_experts(gates, ups, downs, gpu)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)[:, None]
    w = rng.random(ids.shape).astype(np.float32)
    x = torch.from_numpy(rng.standard_normal((len(ids), H)).astype(np.float32)).to(torch.bfloat16)
    xr = x.to(torch.float32).numpy()
    pick = np.sort(rng.permutation(len(ids))[:160])
    ref = oracle.moe_reference(*((lambda b: lambda e: oracle.dequant_q4_1(b[e]))(b) for b in (gates, ups, downs)),
                               xr[pick], ids[pick], w[pick], h_bf16=True)
    for _ in range(2):
        out = pkg.moe_batch(gu, dn, x.to(gpu), ids, w, path="prefill", h_bf16=True).cpu().numpy()
        assert np.isfinite(out).all()
        assert oracle.maxrel(out[pick], ref) <= 1e-3, oracle.maxrel(out[pick], ref)
