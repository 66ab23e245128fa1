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
    "past_wave_long": [(37 * i) % 90 for i in range(64)] + [1100, 0, 3, 261],
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


# Gradient rows outside every sequence are zero, wherever they lie: before the first, behind
# the last, past the longest length, all of them (no sequence at all), and for offsets that
# do not even increase.
@pytest.mark.parametrize("cu,longest", [([40, 90, 90, 300], 210), ([0, 100, 400], 64), ([400, 400], 8),
                                        ([0, 130, 60, 310], 400), ([0], 0)])
def test_varlen_rows_outside_sequences(wo, cu, longest):
    report("varlen_rows_outside_sequences", cu=cu, longest=longest)
    total, h, hkv, d = 400, 4, 2, 64
    g = torch.Generator().manual_seed(9)
    q, do = (torch.randn(total, h, d, generator=g).half().cuda() for _ in range(2))
    k, v = (torch.randn(total, hkv, d, generator=g).half().cuda() for _ in range(2))
    c = torch.tensor(cu, dtype=torch.int32, device="cuda")
    inside = torch.zeros(total, dtype=torch.bool)
    for a, b in zip(cu[:-1], cu[1:]):
        inside[a:min(b, a + longest)] = True
    # two passes over caching-allocator memory that the first left full of NaN
    for _ in range(2):
        o, lse = wo.flash_attention_varlen_forward(q, k, v, c, c, longest, longest, True)
        junk = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        del junk
        grads = wo.flash_attention_varlen_backward(do, q, k, v, o, lse, c, c, longest, longest, True)
        for x in grads:
            assert torch.count_nonzero(x[~inside]) == 0
            assert torch.isfinite(x[~inside]).all()
            if bool(inside.any()):
                assert torch.count_nonzero(x[inside]) > 0


# No query head, or no query row, attends to the keys: their gradients are zero.
@pytest.mark.parametrize("h,total_q", [(0, 30), (4, 0)])
def test_gradients_without_queries(wo, h, total_q):
    report("gradients_without_queries", h=h, total_q=total_q)
    half = dict(dtype=torch.half, device="cuda")
    q, k = torch.zeros(total_q, h, 64, **half), torch.ones(30, 2, 64, **half)
    cq = torch.tensor([0, total_q], dtype=torch.int32, device="cuda")
    ck = torch.tensor([0, 30], dtype=torch.int32, device="cuda")
    for dense in (False, True):
        junk = [torch.full_like(k, float("nan")) for _ in range(8)]
        del junk
        if dense:
            Q, K = q.transpose(0, 1)[None], k.transpose(0, 1)[None]
            O, lse = wo.flash_attention_forward(Q, K, K)
            grads = wo.flash_attention_backward(Q, Q, K, K, O, lse)
        else:
            O, lse = wo.flash_attention_varlen_forward(q, k, k, cq, ck, total_q, 30)
            grads = wo.flash_attention_varlen_backward(q, q, k, k, O, lse, cq, ck, total_q, 30)
        for x in grads:
            assert torch.equal(x, torch.zeros_like(x))


# Many gaps (three times the 64 that one workgroup looks at), and one that is most of a tensor
# larger than one sweep of every workgroup.
@pytest.mark.parametrize("starts,length,total", [(range(3, 3000, 16), 8, 3010), ((5,), 40, 30000)])
def test_varlen_many_and_large_gaps(wo, starts, length, total):
    report("varlen_many_and_large_gaps", total=total)
    h, hkv, d = 4, 2, 64
    cu, longest = list(starts) + [starts[-1] + length], length  # 16 apart, 8 rows of each taken
    g = torch.Generator(device="cuda").manual_seed(13)
    q, do = (torch.randn(total, h, d, generator=g, device="cuda").half() for _ in range(2))
    k, v = (torch.randn(total, hkv, d, generator=g, device="cuda").half() for _ in range(2))
    c = torch.tensor(cu, dtype=torch.int32, device="cuda")
    rows = torch.cat([torch.arange(s, s + length) for s in starts]).cuda()
    near = torch.arange(len(starts) + 1, dtype=torch.int32, device="cuda") * length
    o, lse = wo.flash_attention_varlen_forward(q, k, v, c, c, longest, longest, True)
    on, lsen = wo.flash_attention_varlen_forward(q[rows], k[rows], v[rows], near, near, longest, longest, True)
    junk = [torch.full_like(x, float("nan")) for x in (q, k, v)]
    del junk
    got = wo.flash_attention_varlen_backward(do, q, k, v, o, lse, c, c, longest, longest, True)
    ref = wo.flash_attention_varlen_backward(do[rows], q[rows], k[rows], v[rows], on, lsen, near, near,
                                             longest, longest, True)
    for x, y in zip(got, ref):
        want = torch.zeros_like(x)
        want[rows] = y
        assert torch.equal(x, want)


# Grouped heads over few key blocks: the group's query heads in parts, added per sequence.
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("lens,h,hkv,d", [([300, 0, 77], 8, 2, 64), ([129], 16, 1, 128), ([64, 200], 6, 2, 256)])
def test_varlen_group_parts(wo, lens, h, hkv, d, causal):
    report("varlen_group_parts", lens=lens, h=h, hkv=hkv, d=d, causal=causal)
    g = torch.Generator().manual_seed(11)
    total = sum(lens)
    q, do = (torch.randn(total, h, d, generator=g).half() for _ in range(2))
    k, v = (torch.randn(total, hkv, d, generator=g).half() for _ in range(2))
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    args = (cu.cuda(), cu.cuda(), max(lens), max(lens), causal)
    x = [t.cuda() for t in (q, k, v)]
    o, lse = wo.flash_attention_varlen_forward(*x, *args)
    first = wo.flash_attention_varlen_backward(do.cuda(), *x, o, lse, *args)
    for got, ref in zip(first, oatt.sdpa_varlen_bwd_ref(q, k, v, do, cu, cu, causal)):
        _close(got, ref)
    for got, again in zip(first, wo.flash_attention_varlen_backward(do.cuda(), *x, o, lse, *args)):
        assert torch.equal(got, again)


# The same at batches on both sides of the order's rule (its lines: test_flash_sched.py): the
# parts of a group, whole rows of 32 heads.
@pytest.mark.parametrize("lens,h,hkv,d", [([700, 1300, 40, 300], 16, 2, 128), ([600, 1100, 70], 32, 32, 64),
                                          ([600, 1100, 70, 300], 32, 32, 64)])
@pytest.mark.parametrize("causal", [False, True])
def test_varlen_parts_and_head_rows(wo, lens, h, hkv, d, causal):
    report("varlen_parts_and_head_rows", lens=lens, h=h, hkv=hkv, d=d, causal=causal)
    test_varlen_group_parts(wo, lens, h, hkv, d, causal)
