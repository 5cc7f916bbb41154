"""The routed MoE prefill block where its token rows or its h rows take 2 GiB or more: the expert
GEMMs gather rows through buffer resources of 2^31 - 1 bytes, past which a row would read as
zeros, so such calls go through the per-slot images. A token's result does not depend on the
other tokens, so the last tokens (whose rows lie past 2 GiB) must have the bits they have in a
small batch."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,topk,E,H,F,xdt,precision,h_bf16", [
    (65000, 1, 2, 16640, 128, torch.bfloat16, "bf16", None),     # x rows reach 2.16 GB
    (65000, 1, 2, 16640, 128, torch.bfloat16, "fp16", None),
    (65000, 1, 2, 16640, 128, torch.float32, "fp16", False),     # the same 16-bit rows from f32, two passes
    (65000, 8, 8, 256, 2304, torch.bfloat16, "bf16", None),      # h rows reach 2.4 GB
    (64527, 1, 2, 16640, 128, torch.bfloat16, "fp16", None),     # x just inside 2^31 - 1 bytes: gathered
])
def test_rows_past_2gib(gpu, pkg, oracle, T, topk, E, H, F, xdt, precision, h_bf16):
    say(f"moe prefill large T={T} top{topk} E={E} H={H} F={F} {xdt} {precision}")
    free = torch.cuda.mem_get_info(gpu)[0]
    need = pkg.moe_prefill_workspace_bytes(T, E, topk, H, F) + T * H * 8
    if free < need + (8 << 30):
        pytest.skip(f"{need >> 30} GiB needed")
    rng = np.random.default_rng(H)

    def pack(n, k):
        return pkg.pack_q4_1(oracle.baseline_q4_1_blocks(n, k, rng), gpu)
    gu = pkg.PackedExperts(pack(E * 2 * F, H).data, E, 2 * F, H)
    dn = pkg.PackedExperts(pack(E * H, F).data, E, H, F)
    gen = torch.Generator(gpu).manual_seed(3)
    x = torch.randn(T, H, generator=gen, device=gpu, dtype=xdt)
    ids = torch.randint(0, E, (T, topk), generator=gen, device=gpu, dtype=torch.int32)
    w = torch.rand(T, topk, generator=gen, device=gpu)
    ws = torch.empty(pkg.moe_prefill_workspace_bytes(T, E, topk, H, F), dtype=torch.uint8, device=gpu)
    run = lambda a, b: pkg.moe_batch(gu, dn, x[a:b], ids[a:b], w[a:b], path="prefill", precision=precision,
                                     h_bf16=h_bf16, workspace=ws)
    out = run(0, T)
    for a in (0, T // 2, T - 300):
        assert torch.equal(out[a:a + 300], run(a, a + 300)), f"tokens {a}.. differ from a small batch"
    del out, x, ws
    torch.cuda.empty_cache()
