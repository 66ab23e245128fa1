"""The order in which attention workgroups take their blocks (flash_sched.hpp): every block of
every sequence is computed once, whatever the batch looks like."""
import pytest
import torch

from oracle import attention as oatt
from tests.conftest import report

pytestmark = pytest.mark.gpu

BAR = 1e-3  # max |got - ref| / max |ref|, the bar of every attention test


def _close(got, ref):
    err = (got.float().cpu() - ref.float()).abs().max() / ref.float().abs().max()
    assert err <= BAR, float(err)


# Fewer and more sequences than a wave has lanes, empty ones, blocks that end one row short of
# or past a tile, head counts on both sides of the 8 XCDs and the 32 engines.
BATCHES = {
    "one": [700],
    "edges": [256, 255, 257, 1, 128, 129, 127],
    "empty": [0, 300, 0, 0, 65, 0],
    "wave": [17] * 63 + [520],
    "past_wave": [(37 * i) % 90 for i in range(64)] + [400, 0, 3, 261],
    "long": [700, 1500, 90, 0, 1000, 1281],
    "two_waves": [(11 * i) % 23 for i in range(130)] + [300],
}


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,hkv,d", [(1, 1, 64), (3, 1, 128), (8, 8, 64), (40, 8, 64), (2, 2, 256)])
@pytest.mark.parametrize("name", sorted(BATCHES))
def test_varlen_every_block_once(wo, name, h, hkv, d, causal):
    lens = BATCHES[name]
    g = torch.Generator().manual_seed(5)
    total = sum(lens)
    q, do = (torch.randn(total, h, d, generator=g).half() for _ in range(2))
    k, v = (torch.randn(total, hkv, d, generator=g).half() for _ in range(2))
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    args = (cu.cuda(), cu.cuda(), max(lens), max(lens))
    report("varlen_every_block_once", batch=name, h=h, hkv=hkv, d=d, causal=causal)
    leaves = [x.cuda().requires_grad_(True) for x in (q, k, v)]
    o = wo.flash_attention_varlen(*leaves, *args, causal=causal)
    grads = torch.autograd.grad(o, leaves, do.cuda())
    _close(o.detach(), oatt.sdpa_varlen_ref(q, k, v, cu, cu, causal))
    for got, ref in zip(grads, oatt.sdpa_varlen_bwd_ref(q, k, v, do, cu, cu, causal)):
        _close(got, ref)
