"""GEMM operands read in the storage order of a view: transposes and column slices."""
import pytest
import torch

from oracle import gemm as og
from tests.conftest import report

pytestmark = pytest.mark.gpu

BAR = 1e-4  # max |got - ref| / max |ref|: fp32 sums on both sides


def _close(got, ref):
    err = (got.cpu() - ref).abs().max() / ref.abs().max().clamp_min(1e-30)
    assert err <= BAR, float(err)


def _inputs(m, n, k, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(m, k, generator=g).half(), torch.randn(k, n, generator=g).half()


def _stored_transposed(x):
    return x.t().contiguous().cuda().t()


# Tile edges and remainders in each dimension; the skinny kernel's row blocks, column counts
# and K rounds (8 x 128 per workgroup); rows that are not whole 16-byte vectors, which the
# skinny kernel reads in place (odd K: rows start at odd elements) and the others copy.
SHAPES = [
    (1, 16, 8), (1, 77, 30), (3, 515, 1), (16, 4096, 1024), (16, 300, 1032), (5, 983, 589),
    (17, 64, 2051), (31, 1000, 2050), (32, 2048, 4096), (33, 96, 72), (64, 64, 64), (65, 136, 200),
    (127, 250, 333), (256, 256, 256), (257, 264, 520), (787, 983, 589), (1000, 4100, 1032),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("which", ["a", "b", "ab"])
def test_transposed_views(wo, m, n, k, which):
    report("transposed_views", m=m, n=n, k=k, which=which)
    A, B = _inputs(m, n, k)
    a = _stored_transposed(A) if "a" in which else A.cuda()
    b = _stored_transposed(B) if "b" in which else B.cuda()
    ref = og.gemm_ref(A, B)
    got = wo.matmul(a, b)
    _close(got, ref)
    assert torch.equal(got, wo.matmul(a, b))
    C = torch.randn(m, n, generator=torch.Generator().manual_seed(3))
    _close(wo.gemm(a, b, 2.0, 0.5, C.cuda()), og.gemm_ref(A, B, 2.0, 0.5, C))
    Ci = C.cuda()
    wo.gemm_inplace(a, b, Ci, 2.0, 0.5)
    _close(Ci, og.gemm_ref(A, B, 2.0, 0.5, C))


@pytest.mark.parametrize("tile", range(6))
@pytest.mark.parametrize("which", ["a", "b"])
def test_transposed_every_tile(wo, tile, which):
    m, n, k = 520, 328, 136
    report("transposed_every_tile", tile=tile, which=which)
    A, B = _inputs(m, n, k, 1)
    a = _stored_transposed(A) if which == "a" else A.cuda()
    b = _stored_transposed(B) if which == "b" else B.cuda()
    # the same products in the same order as on contiguous copies
    assert torch.equal(wo.matmul_tiled(a, b, tile), wo.matmul_tiled(A.cuda(), B.cuda(), tile))
    _close(wo.matmul_tiled(a, b, tile), og.gemm_ref(A, B))


@pytest.mark.parametrize("off", [0, 1, 2, 3, 8])
@pytest.mark.parametrize("m", [4, 20, 150])
def test_sliced_views(wo, m, off):
    # Slices keep their parent's stride: rows at any element offset, and a parent whose row
    # length is odd, plain and transposed.
    report("sliced_views", m=m, off=off)
    g = torch.Generator().manual_seed(2)
    X, W = torch.randn(m, 521, generator=g).half(), torch.randn(512, 331, generator=g).half()
    Wt = torch.randn(300, 533, generator=g).half()
    a, A = X.cuda()[:, off:off + 512], X[:, off:off + 512]
    b, B = W.cuda()[:, off:off + 300], W[:, off:off + 300]
    _close(wo.matmul(a, b), og.gemm_ref(A, B))
    bt, Bt = Wt.cuda()[:, off:off + 512].t(), Wt[:, off:off + 512].t()
    _close(wo.matmul(a, bt), og.gemm_ref(A, Bt))


def test_other_strides_are_copied(wo):
    # Steps, expanded rows and strides past the kernels' 32-bit offsets.
    A, B = _inputs(48, 40, 64, 4)
    ref = og.gemm_ref(A, B)
    wide = torch.zeros(48, 128, dtype=torch.half, device="cuda")
    wide[:, ::2] = A.cuda()
    _close(wo.matmul(wide[:, ::2], B.cuda()), ref)
    row = torch.randn(1, 64).half()
    _close(wo.matmul(row.cuda().expand(48, 64), B.cuda()), og.gemm_ref(row.expand(48, 64), B))
    far = torch.empty(2 * 5000000, dtype=torch.half, device="cuda").as_strided((2, 64), (5000000, 1))
    far.copy_(A[:2])
    _close(wo.matmul(far, B.cuda()), ref[:2])
    _close(wo.matmul(B.cuda().t(), far.t()), og.gemm_ref(B.t(), A[:2].t()))


# Two-part plans of each layout: an edge of the transposed B's streaming kernel with a K split
# (its workspace is not that of the plain layout's edge) and without one, of the tiled kernel,
# of rows and of columns.
@pytest.mark.parametrize("m,n,k", [(1300, 11008, 4096), (2840, 11008, 4096), (4100, 4096, 1024),
                                   (2848, 11008, 4096), (4096, 4104, 1024), (785, 18944, 3584)])
def test_transposed_two_part(wo, m, n, k):
    report("transposed_two_part", m=m, n=n, k=k)
    g = torch.Generator(device="cuda").manual_seed(6)
    a = torch.randn(m, k, generator=g, device="cuda").half()
    w = torch.randn(n, k, generator=g, device="cuda").half()
    C = torch.randn(m, n, generator=g, device="cuda")
    ref = a.float() @ w.float().t()
    at = a.t().contiguous().t()
    for x, y in ((a, w.t()), (at, w.t().contiguous())):
        _close(wo.matmul(x, y), ref.cpu())
        _close(wo.gemm(x, y, 2.0, 0.5, C), (2.0 * ref + 0.5 * C).cpu())
        out = C.clone()
        wo.gemm_inplace(x, y, out, 2.0, 0.5)
        _close(out, (2.0 * ref + 0.5 * C).cpu())


def test_one_row_at_any_stride(wo):
    # A contiguous tensor of one row may carry any row stride: the transpose of a column has 1.
    g = torch.Generator().manual_seed(8)
    B, W = torch.randn(96, 200, generator=g).half(), torch.randn(200, 1, generator=g).half()
    col, C = torch.randn(96, 1, generator=g).half(), torch.randn(200, 1, generator=g)
    x = torch.randn(50, 1, generator=g).half()
    ref = og.gemm_ref(col.t(), B)
    report("one_row_at_any_stride", strides=col.t().stride())
    _close(wo.matmul(col.cuda().t(), B.cuda()), ref)
    far = torch.empty(96, dtype=torch.half, device="cuda").as_strided((1, 96), (1 << 40, 1))
    far.copy_(col.t())
    _close(wo.matmul(far, B.cuda()), ref)
    _close(wo.matmul(x.cuda(), W.cuda().t()), og.gemm_ref(x, W.t()))           # B [1, N]
    _close(wo.matmul_tiled(x.cuda(), W.cuda().t(), 0), og.gemm_ref(x, W.t()))
    ref = og.gemm_ref(col.t(), B, 2.0, 0.5, C.t())
    _close(wo.gemm(col.cuda().t(), B.cuda(), 2.0, 0.5, C.cuda().t()), ref)
    out = C.cuda().t()
    wo.gemm_inplace(col.cuda().t(), B.cuda(), out, 2.0, 0.5)
    _close(out, ref)


def test_int4_one_row_at_any_stride(wo):
    g = torch.Generator().manual_seed(9)
    q = torch.randint(-2 ** 31, 2 ** 31, (32, 64), generator=g, dtype=torch.int64).int().cuda()
    s = (torch.rand(2, 64, generator=g) * 0.01).half().cuda()
    z = torch.randint(0, 16, (2, 64), generator=g, dtype=torch.uint8).cuda()
    a = torch.randn(256, 1, generator=g).half().cuda()
    row = a.reshape(1, 256).clone()
    p, f = wo.prepack_int4(q), wo.prepack_int4_fused(q, s, z, 128)
    assert torch.equal(wo.matmul_int4(a.t(), p, s, z, 128), wo.matmul_int4(row, p, s, z, 128))
    assert torch.equal(wo.matmul_int4_fused(a.t(), f, 128), wo.matmul_int4_fused(row, f, 128))


def test_inplace_on_a_view_of_c(wo):
    # A strided fp16 view of C's own memory is read before C is written: more tiles than run at
    # once, each row of tiles writing over the A of the next.
    report("inplace_on_a_view_of_c")
    m, n, k = 4096, 5120, 4096
    g = torch.Generator(device="cuda").manual_seed(10)
    halves = torch.randn(m, 2 * n, generator=g, device="cuda").half()
    b = torch.randn(k, n, generator=g, device="cuda").half()
    a, c = halves[:, 512:512 + k], halves.view(torch.float32)
    assert c.shape == (m, n) and c.isfinite().all()
    ref = wo.gemm(a.contiguous(), b, 2.0, 0.5, c.clone())
    wo.gemm_inplace(a, b, c, 2.0, 0.5)
    assert torch.equal(c, ref)
    bt = torch.randn(n, 2 * m, generator=g, device="cuda").half()  # C^T: B a view of it
    c, b = bt.view(torch.float32), bt[:, :m]
    a = torch.randn(n, n, generator=g, device="cuda").half()
    ref = wo.gemm(a, b.contiguous(), 2.0, 0.5, c.clone())
    wo.gemm_inplace(a, b, c, 2.0, 0.5)
    assert torch.equal(c, ref)


def test_repack_past_one_launch(wo):
    # Rows off 16 bytes whose copy is more 16-byte chunks than one grid has threads (2^32).
    m, k = 8300, 4177973
    if torch.cuda.mem_get_info()[0] < 180 << 30:
        pytest.skip("needs 180 GiB of GPU memory")
    report("repack_past_one_launch", m=m, k=k)
    a = torch.ones(m, k, dtype=torch.half, device="cuda")
    a[m // 2] = 2
    a[-1, 1::2] = 3
    b = torch.ones(k, 8, dtype=torch.half, device="cuda")
    got = wo.matmul(a, b)
    ref = torch.full((m, 8), float(k), device="cuda")  # whole numbers below 2^24
    ref[m // 2] = 2 * k
    ref[-1] = k + 2 * (k // 2)
    assert torch.equal(got, ref)
    del a, b
    torch.cuda.empty_cache()
