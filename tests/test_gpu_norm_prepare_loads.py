"""q4_rmsnorm_prepare's loads: rows at the ends of each instance's range, plane counts around the
batch the loads go out in, and pointers that are only 4-byte aligned (16-byte loads are then not
taken). The oracle is the row added up in the documented order with torch, then rmsnorm_add
and prefill_prepare: the same bytes."""
from __future__ import annotations

import pytest
import torch

from conftest import say

pytestmark = pytest.mark.gpu


def _rows(gpu, T, K, shift, seed):
    g = torch.Generator(gpu).manual_seed(seed)
    buf = torch.randn(T * K + 4, generator=g, device=gpu)
    return buf[shift:shift + T * K].view(T, K)


def _check(gpu, pkg, T, K, planes, shift, wdt):
    x = _rows(gpu, T, K, shift, 1)
    add = _rows(gpu, planes * T, K, shift, 2).view(planes, T, K) if planes else None
    w = _rows(gpu, 1, K, shift, 3).view(-1).to(wdt)
    if shift:
        w = torch.cat([w[:1], w])[1:]                     # off 16 bytes as well
    y = torch.empty(T * K + 4, device=gpu)[shift:shift + T * K].view(T, K)
    nbytes = int(pkg.load_library().q4_prefill_prepared_bytes(T, K, 1, 0))
    zeros = lambda: torch.zeros(nbytes, dtype=torch.uint8, device=gpu)
    got_y, got = pkg.rmsnorm_prepare(x, w, add=add, y=y, out=zeros())
    ref_y = x
    if planes:
        s = add[0]
        for q in range(1, planes):
            s = s + add[q]
        ref_y = x + s
    _, xn = pkg.rmsnorm_add(ref_y.contiguous().clone(), w.clone(), out_dtype=torch.bfloat16)
    ref = pkg.prefill_prepare(xn, out=zeros())
    torch.cuda.synchronize()
    assert torch.equal(got_y, ref_y)
    assert torch.equal(got.data, ref.data)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("K", [32, 992, 1024, 1056, 2048, 2080, 4096, 4128, 8192, 8224, 16384])
@pytest.mark.parametrize("planes", [0, 1, 2, 4, 5, 9])
@pytest.mark.parametrize("wdt", [torch.bfloat16, torch.float32])
def test_planes_and_alignment(gpu, pkg, K, planes, shift, wdt):
    say(f"rmsnorm_prepare loads K={K} planes={planes} shift={shift} {wdt}")
    _check(gpu, pkg, 3, K, planes, shift, wdt)


# 48 MiB of planes and one row more: loaded together, then one behind the other
@pytest.mark.parametrize("K,planes", [(1024, 6), (2048, 3), (4096, 2), (8192, 3), (16384, 2)])
@pytest.mark.parametrize("more", [0, 1])
def test_planes_past_the_caches(gpu, pkg, K, planes, more):
    T = (48 << 20) // (planes * K * 4) + more
    say(f"rmsnorm_prepare loads T={T} K={K} planes={planes}")
    _check(gpu, pkg, T, K, planes, 0, torch.bfloat16)
