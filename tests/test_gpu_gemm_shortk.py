"""Products of many outputs over a K slab or two, against float64: ragged tiles, whole and ragged slabs, K segments, groups, addend,
row sums and the fused update; and against the order of sums of the kernels they had before."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


def _run(dtype, a, b, m, n, k, akc, bkc, **kw):
    from rtp_amd import _lib, ops
    _lib.profile_enable(1)
    try:
        done = ops.gemm_raw(dtype, a=a.data_ptr(), b=b.data_ptr(), m=m, n=n, k=k, a_kcontig=akc, b_kcontig=bkc, **kw)
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    assert any("shortk" in nm for nm in names), names
    return done


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("akc,bkc", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("m,n,k,ksegs,groups", [(2568, 2392, 8, 1, 1), (136, 1032, 24, 1, 22), (264, 2056, 64, 1, 8), (8, 136, 16, 2, 200),
                                                (1544, 4104, 32, 2, 1)])
def test_edges(dtype, akc, bkc, m, n, k, ksegs, groups):
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(ksegs, groups, m, k, generator=gen).to(dtype).to(DEV)
    b = torch.randn(ksegs, groups, n, k, generator=gen).to(dtype).to(DEV)
    cin = torch.randn(groups, m, n, generator=gen).to(dtype).to(DEV)
    # NaN behind the last row and column: nothing of it may reach a result
    A = torch.full((ksegs, groups, m, k + 8) if akc else (ksegs, groups, k, m + 8), float("nan"), dtype=dtype, device=DEV)
    B = torch.full((ksegs, groups, n, k + 8) if bkc else (ksegs, groups, k, n + 8), float("nan"), dtype=dtype, device=DEV)
    A[..., :k if akc else m] = a if akc else a.transpose(2, 3)
    B[..., :k if bkc else n] = b if bkc else b.transpose(2, 3)
    out = torch.full((groups, m, n), float("nan"), dtype=dtype, device=DEV)
    sums = torch.full((groups, m), float("nan"), dtype=dtype, device=DEV)
    done = _run(dtype, A, B, m, n, k, akc, bkc, c_out=out.data_ptr(), lda=A.stride(2), ldb=B.stride(2), ldc=n, groups=groups,
                a_sg=A.stride(1), b_sg=B.stride(1), c_sg=m * n, ksegs=ksegs, a_sk=A.stride(0), b_sk=B.stride(0),
                c_in=cin.data_ptr(), ld_cin=n, cin_sg=m * n, rowsum=None if akc else sums.data_ptr(), rowsum_sg=m)
    # one rounding of 2^-24 per product, one for the addend; the result's own
    own = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    for g in range(groups):
        x, y = a[:, g].double(), b[:, g].double()
        ref = torch.stack([x[s] @ y[s].t() for s in range(ksegs)]).sum(0) + cin[g].double()
        size = torch.stack([x[s].abs() @ y[s].abs().t() for s in range(ksegs)]).sum(0) + cin[g].double().abs()
        assert ((out[g].double() - ref).abs() <= (ksegs * k + 1) * 2.0 ** -24 * size + own * ref.abs()).all(), g
        if done:
            rows, size = x.sum((0, 2)), x.abs().sum((0, 2))
            assert ((sums[g].double() - rows).abs() <= ksegs * k * 2.0 ** -24 * size + own * rows.abs()).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_update_and_order(dtype):
    """clip + SGD in the epilogue is bit for bit the update by the gradient the product without it stores; and that gradient has the
    bits of the same rows computed as a product of fewer tiles, by another kernel."""
    from rtp_amd import ops
    m, n, k = 2560, 2560, 40
    gen = torch.Generator().manual_seed(2)
    a, b = (torch.randn(k, c, generator=gen).to(dtype).to(DEV) for c in (m, n))
    w = torch.randn(m, n, generator=gen).to(DEV)
    grad, kept, master, copy = (torch.zeros(m, n, dtype=t, device=DEV) for t in (dtype, dtype, torch.float32, dtype))
    master.copy_(w)
    common = dict(lda=m, ldb=n, ldc=n)
    _run(dtype, a, b, m, n, k, False, False, c_out=grad.data_ptr(), **common)
    sgd = ops.FusedSgd(lr=0.1, clip=5.0, keep_grads=True)
    _run(dtype, a, b, m, n, k, False, False, c_out=kept.data_ptr(), sgd=sgd, sgd_master=master.data_ptr(),
         sgd_weights=copy.data_ptr() if dtype == torch.bfloat16 else 0, **common)
    assert not sgd.missed and torch.equal(kept, grad) and float(grad.abs().max()) > 5.0
    assert torch.equal(master, w - 0.1 * grad.float().clamp(-5.0, 5.0))
    if dtype == torch.bfloat16:
        assert torch.equal(copy, master.to(dtype))
    part = torch.zeros(1280, n, dtype=dtype, device=DEV)
    ops.gemm_raw(dtype, a=a.data_ptr(), b=b.data_ptr(), c_out=part.data_ptr(), m=1280, n=n, k=k, a_kcontig=False, b_kcontig=False,
                 **common)
    assert torch.equal(part, grad[:1280])
