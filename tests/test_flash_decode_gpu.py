"""The decoding kernel (flash_decode.hip): at most 32 query rows per key/value head, no mask."""
import ctypes
import math

import pytest
import torch

from oracle import attention as oatt
from oracle import gemm as og
from tests.conftest import report

pytestmark = pytest.mark.gpu


def _case(wo, B, H, Hkv, Sq, Sk, D, scale=-1.0, spread=1.0):
    Q, K, V = oatt.make_inputs(B, H, Sq, D, seed=Sk + D, Sk=Sk, Hkv=Hkv)
    Q = (Q.float() * spread).half()
    O, lse = wo.flash_attention_forward(Q.cuda(), K.cuda(), V.cuda(), False, scale)
    assert og.max_rel_err(O.float().cpu(), oatt.sdpa_ref(Q, K, V, False, scale)) <= 1e-3
    lref = oatt.lse_ref(Q, K, False, scale)
    assert torch.allclose(lse.cpu(), lref, atol=1e-3, rtol=1e-5)
    assert torch.equal(wo.flash_attention(Q.cuda(), K.cuda(), V.cuda(), False, scale), O)
    return O


# Keys: one, around a step (32), around one step per wave (128) and a split; rows per
# key/value head: 1, both sides of a 16-row block, the most (32) and one more (the general
# kernel, which also takes over 16 rows against at most 128 keys at D > 64); every head-dim
# kernel and head dims that do not fill it.
@pytest.mark.parametrize("Sk", [1, 31, 33, 127, 128, 129, 260, 1025, 5000])
@pytest.mark.parametrize("H,Hkv,Sq", [(2, 2, 1), (15, 1, 1), (8, 1, 2), (17, 1, 1), (8, 1, 4), (33, 1, 1)])
def test_decode_rows_and_keys(wo, H, Hkv, Sq, Sk):
    report("decode_rows_and_keys", H=H, Hkv=Hkv, Sq=Sq, Sk=Sk)
    _case(wo, 2, H, Hkv, Sq, Sk, 128)


@pytest.mark.parametrize("D", [8, 40, 64, 72, 100, 128, 136, 200, 256])
@pytest.mark.parametrize("H,Hkv,Sq", [(4, 2, 1), (20, 1, 1)])
@pytest.mark.parametrize("Sk", [77, 3001])
def test_decode_head_dims(wo, D, H, Hkv, Sq, Sk):
    report("decode_head_dims", D=D, H=H, Hkv=Hkv, Sq=Sq, Sk=Sk)
    _case(wo, 1, H, Hkv, Sq, Sk, D)


def test_decode_growing_maximum(wo):
    # Scores that grow along the keys (each step's above the last by more than the running
    # maximum's slack) and a wide score range: the rescaling path, in one chunk and several.
    for Sk in (300, 6000):
        report("decode_growing_maximum", Sk=Sk)
        D = 128
        Q = torch.ones(1, 2, 1, D).half()
        K = (torch.arange(Sk).float() / Sk * 4).view(1, 1, Sk, 1).expand(1, 2, Sk, D).half()
        V = torch.randn(1, 2, Sk, D, generator=torch.Generator().manual_seed(1)).half()
        O = wo.flash_attention(Q.cuda(), K.contiguous().cuda(), V.cuda(), False)
        assert og.max_rel_err(O.float().cpu(), oatt.sdpa_ref(Q, K, V, False)) <= 1e-3
    _case(wo, 2, 8, 2, 4, 2050, 64, spread=8.0)
    _case(wo, 1, 4, 4, 3, 515, 128, scale=1.0 / math.sqrt(7))


def _one_pass(wo, Q, K, V):
    # without a workspace the key range is never split
    L = ctypes.CDLL(wo.LIBRARY_PATH)
    vp, i32 = ctypes.c_void_p, ctypes.c_int
    L.wmma_flash_attn_fwd_lse.argtypes = [vp] * 5 + [i32] * 6 + [ctypes.c_float, i32, vp]
    (B, H, Sq, D), (Hkv, Sk) = Q.shape, K.shape[1:3]
    O, lse = torch.empty_like(Q), torch.empty(B, H, Sq, device="cuda")
    assert L.wmma_flash_attn_fwd_lse(Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(),
                                     lse.data_ptr(), B, H, Hkv, Sq, Sk, D, 1.0 / math.sqrt(D), 0,
                                     torch.cuda.current_stream().cuda_stream) == 0
    return O, lse


# One chunk of keys and several, on the decoding kernel and (64 rows) the general one.
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk", [(160, 1, 1, 1, 64), (160, 1, 1, 1, 4096), (2, 8, 2, 1, 5000),
                                           (1, 2, 1, 32, 4096)])
@pytest.mark.parametrize("what", ["query", "keys", "all keys", "values", "infinite keys"])
def test_decode_nan(wo, B, H, Hkv, Sq, Sk, what):
    # A NaN reaches the rows that it reaches in one pass over the keys, wherever the chunks lie.
    report("decode_nan", B=B, H=H, Hkv=Hkv, Sq=Sq, Sk=Sk, what=what)
    Q, K, V = (t.cuda() for t in oatt.make_inputs(B, H, Sq, 64, seed=7, Sk=Sk, Hkv=Hkv))
    if what == "query":
        Q[0, -1, Sq // 2, 3] = math.nan
    elif what == "values":
        V[0, 0, Sk // 2, 5] = math.nan
    else:
        n = Sk if what == "all keys" else max(Sk // 4, 1)
        K[0, 0, :n, 1] = math.inf if what == "infinite keys" else math.nan
    O, lse = wo.flash_attention_forward(Q, K, V, False)
    O1, lse1 = _one_pass(wo, Q, K, V)
    assert O1.isnan().any()
    assert torch.equal(O.isnan(), O1.isnan())
    assert torch.equal(lse.isnan(), lse1.isnan())
    assert torch.allclose(lse, lse1, atol=1e-3, rtol=1e-5, equal_nan=True)
    assert torch.allclose(O.float(), O1.float(), atol=2e-3, rtol=0, equal_nan=True)
    assert torch.equal(wo.flash_attention(Q, K, V, False).isnan(), O1.isnan())
