"""Groups of 32 and 64 at M <= 32: the decode, skinny and rows kernels with a scale and zero
per lane.  They form fp16((q - z) s) per weight, so only the order of the fp32 sum differs
from the oracle; 1e-3 is the output tolerance of the path."""
import numpy as np
import pytest
import torch

from oracle import gemm as og
from oracle import int4 as oi
from tests.conftest import report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zeros", ["packed", "bytes", "sliced"])
@pytest.mark.parametrize("G", [32, 64])
# K: one pair-step, a last round that is not full, one past the decode kernel's single round,
# and long enough for a K split
@pytest.mark.parametrize("N,K", [(32, 128), (96, 1152), (1024, 4224), (256, 11008), (4096, 2048)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 17, 32])
def test_fine_groups(wo, M, N, K, G, zeros):
    plan = wo.w4a16_plan(M, N, K, G)
    report("w4a16_fine_groups", M=M, N=N, K=K, G=G, zeros=zeros, plan=plan)
    assert plan[0] in ((0, 4) if M <= 4 else (4, 6))  # decode; skinny; rows
    A, q, s, z = oi.make_inputs(M, K, N, G, seed=M + K + G)
    pk = wo.prepack_int4(torch.from_numpy(oi.pack_gptq(q)).cuda())
    sd, zd = torch.from_numpy(s).cuda(), torch.from_numpy(oi.pack_zeros(z)).cuda()
    if zeros == "bytes":
        zd = torch.from_numpy(np.ascontiguousarray(z).astype(np.uint8)).cuda()
    if zeros == "sliced":
        sd, zd = wo.prepack_int4_params(sd, zd)
    assert og.max_rel_err(wo.matmul_int4(A.cuda(), pk, sd, zd, G),
                          oi.w4a16_ref(A, q, s, z, G)) <= 1e-3
