"""Attention on views: every storage order gives what contiguous copies give."""
import pytest
import torch

from tests.conftest import report

pytestmark = pytest.mark.gpu


def _gen(seed):
    return torch.Generator().manual_seed(seed)


def _bshd(b, h, s, d, seed):
    """[b, h, s, d] as the transposed view of a projection's [b, s, h * d] output."""
    return torch.randn(b, s, h * d, generator=_gen(seed)).half().cuda().view(b, s, h, d).transpose(1, 2)


def _qkv(b, h, s, d, seed):
    """Three [b, h, s, d] slices of one fused [b, s, 3, h, d] projection."""
    x = torch.randn(b, s, 3, h, d, generator=_gen(seed)).half().cuda()
    return [x[:, :, i].transpose(1, 2) for i in range(3)]


def _step(wo, q, k, v, do, causal):
    leaves = [x.detach().requires_grad_(True) for x in (q, k, v)]
    assert leaves[0].stride() == q.stride()
    o = wo.flash_attention(*leaves, causal=causal)
    return (o.detach(), *torch.autograd.grad(o, leaves, do))


def _same(got, want):
    for g, w in zip(got, want):
        assert g.is_contiguous() and torch.equal(g, w)


# Causal and not; grouped heads (packed by a copy of Q where single heads waste blocks, run
# head by head where they do not); one query; head dims that are padded, or fill no kernel.
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,hkv,sq,sk,d", [
    (2, 4, 4, 300, 300, 128), (1, 8, 2, 513, 513, 64), (2, 6, 3, 77, 100, 128),
    (2, 8, 2, 1, 700, 128), (1, 16, 2, 3, 1500, 64), (3, 5, 1, 130, 64, 80), (1, 2, 2, 65, 65, 100),
    (2, 2, 1, 200, 140, 256), (1, 1, 1, 90, 90, 72)])
def test_projection_views(wo, b, h, hkv, sq, sk, d, causal):
    report("projection_views", b=b, h=h, hkv=hkv, sq=sq, sk=sk, d=d, causal=causal)
    q, k, v, do = (_bshd(b, n, s, d, i) for i, (n, s) in enumerate([(h, sq), (hkv, sk), (hkv, sk), (h, sq)]))
    plain = [x.contiguous() for x in (q, k, v, do)]
    _same(_step(wo, q, k, v, do, causal), _step(wo, *plain, causal))
    assert torch.equal(wo.flash_attention(q, k, v, causal), wo.flash_attention(*plain[:3], causal))


def test_fused_projection_and_mixed_strides(wo):
    report("fused_projection_and_mixed_strides")
    b, h, s, d = 2, 4, 260, 64
    q, k, v = _qkv(b, h, s, d, 3)
    do = _bshd(b, h, s, d, 4)  # another row stride than q's
    plain = [x.contiguous() for x in (q, k, v, do)]
    _same(_step(wo, q, k, v, do, True), _step(wo, *plain, True))
    _same(_step(wo, plain[0], k, plain[2], do, True), _step(wo, *plain, True))
    # one cache for every batch entry, read at stride 0
    ke, ve = (x[:1].expand(b, h, s, d) for x in (plain[1], plain[2]))
    want = wo.flash_attention(plain[0], ke.contiguous(), ve.contiguous())
    assert torch.equal(wo.flash_attention(q, ke, ve), want)
    # rows off 16-byte vectors and a stepped last dimension are copied
    wide = torch.randn(b, h, s, d + 4, generator=_gen(5)).half().cuda()
    for view in (wide[..., :d], wide[..., 2:d + 2]):
        assert torch.equal(wo.flash_attention(view, k, v), wo.flash_attention(view.contiguous(), *plain[1:3]))
    step = torch.randn(b, h, s, 2 * d, generator=_gen(6)).half().cuda()[..., ::2]
    assert torch.equal(wo.flash_attention(q, step, v), wo.flash_attention(plain[0], step.contiguous(), plain[2]))


@pytest.mark.parametrize("causal", [False, True])
def test_packed_views(wo, causal):
    report("packed_views", causal=causal)
    h, d, lens = 4, 128, [70, 0, 300, 129]
    total = sum(lens)
    x = torch.randn(total, 3, h, d, generator=_gen(7)).half().cuda()
    q, k, v = (x[:, i] for i in range(3))
    do = torch.randn(h, total, d, generator=_gen(8)).half().cuda().transpose(0, 1)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()

    def step(q, k, v, do):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o = wo.flash_attention_varlen(*leaves, cu, cu, max(lens), max(lens), causal=causal)
        return (o.detach(), *torch.autograd.grad(o, leaves, do))

    want = step(*(t.contiguous() for t in (q, k, v, do)))
    _same(step(q, k, v, do), want)                # Q and dO at different row strides
    do2 = torch.empty(total, 3, h, d, dtype=torch.half, device="cuda")[:, 1].copy_(do)
    _same(step(q, k, v, do2), want)               # every tensor in place
