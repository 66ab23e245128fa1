"""Head dims around 96, where the kernel changes: forward and backward against the oracle."""
import pytest
import torch

from oracle import attention as oatt
from oracle import gemm as og
from tests.conftest import report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [64, 65, 72, 88, 96, 97, 104])
@pytest.mark.parametrize("H,Hkv,Sq,Sk", [(2, 1, 300, 260), (4, 4, 65, 65)])
def test_head_dims_around_96(wo, D, H, Hkv, Sq, Sk, causal):
    report("head_dims_around_96", D=D, H=H, Hkv=Hkv, Sq=Sq, Sk=Sk, causal=causal)
    Q, K, V = oatt.make_inputs(2, H, Sq, D, seed=D + Sq, Sk=Sk, Hkv=Hkv)
    dO = torch.randn(Q.shape, generator=torch.Generator().manual_seed(D)).half()
    leaves = [x.cuda().requires_grad_(True) for x in (Q, K, V)]
    O = wo.flash_attention(*leaves, causal=causal)
    grads = torch.autograd.grad(O, leaves, dO.cuda())
    assert og.max_rel_err(O.detach().float().cpu(), oatt.sdpa_ref(Q, K, V, causal)) <= 1e-3
    for got, ref in zip(grads, oatt.sdpa_bwd_ref(Q, K, V, dO, causal)):
        assert og.max_rel_err(got.float().cpu(), ref) <= 1e-3
