"""The VALU decode kernel (M <= 4, groups that are not 32 * 2^j) at activations that do not
fill its staging rounds of 512 16-byte chunks."""
import numpy as np
import pytest
import torch

from oracle import gemm as og
from oracle import int4 as oi
from tests.conftest import report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zeros", ["packed", "bytes", "sliced"])
@pytest.mark.parametrize("K", [384, 1152, 1920, 4224, 5376])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_w4a16_decode_partial_staging(wo, M, K, zeros):
    N, G = 4096, 96
    plan = wo.w4a16_plan(M, N, K, G)
    report("w4a16_decode_partial_staging", M=M, K=K, zeros=zeros, plan=plan)
    assert plan[0] == 1
    A, q, s, z = oi.make_inputs(M, K, N, G, seed=M + K)
    pk = wo.prepack_int4(torch.from_numpy(oi.pack_gptq(q)).cuda())
    sd, zd = torch.from_numpy(s).cuda(), torch.from_numpy(oi.pack_zeros(z)).cuda()
    if zeros == "bytes":
        zd = torch.from_numpy(np.ascontiguousarray(z).astype(np.uint8)).cuda()
    if zeros == "sliced":
        sd, zd = wo.prepack_int4_params(sd, zd)
    first = wo.matmul_int4(A.cuda(), pk, sd, zd, G)
    assert og.max_rel_err(first, oi.w4a16_ref(A, q, s, z, G)) <= 1e-3
    for _ in range(3):
        assert torch.equal(wo.matmul_int4(A.cuda(), pk, sd, zd, G), first)
