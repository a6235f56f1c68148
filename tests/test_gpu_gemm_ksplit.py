"""fp32 products of row-contiguous operands with few tiles and a long contraction (the contraction split over the waves of a
workgroup), against float64: contractions that leave waves without work or with a ragged batch, ragged tiles, groups, K
segments, an addend, a bias and row sums.  Bound: fp32 sums of up to 3000 products, 1e-5 of the largest result."""
import pytest
import torch

from test_gpu_gemm import DEV, TOL, _ops, _rand, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,groups,segs", [(512, 512, 1600, 1, 1), (32, 32, 512, 1, 1), (33, 31, 513, 1, 1), (64, 100, 527, 4, 1),
                                               (5, 700, 2881, 1, 1), (512, 260, 640, 1, 3), (1, 8, 1000, 1, 1)])
@pytest.mark.parametrize("accum", [False, True])
def test_split_contraction(m, n, k, groups, segs, accum):
    from rtp_amd import _lib
    gen = torch.Generator().manual_seed(m + n + k)
    lda, ldb = m + 3, n + 1  # no alignment needed
    a = _rand((segs, groups, k, lda), torch.float32, gen)
    b = _rand((segs, groups, k, ldb), torch.float32, gen)
    cin, bias = _rand((groups, m, n), torch.float32, gen), _rand((groups, n), torch.float32, gen)
    A, B = a[..., :m].double(), b[..., :n].double()
    ref = (A.transpose(2, 3) @ B).sum(0)
    rows = A.sum((0, 2))
    if accum:
        ref = ref + cin.double() + bias.double()[:, None]
    ad, bd, cd, bias_d = (t.to(DEV) for t in (a, b, cin, bias))
    out = torch.full((groups, m, n), float("nan"), device=DEV)
    sums = torch.full((groups, m), float("nan"), device=DEV)
    extra = dict(c_in=cd.data_ptr(), ld_cin=n, cin_sg=m * n, bias=bias_d.data_ptr(), bias_sg=n) if accum else {}
    _lib.profile_enable(1)
    try:
        fused = _ops().gemm_raw(torch.float32, a=ad.data_ptr(), b=bd.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=lda,
                                ldb=ldb, ldc=n, a_kcontig=False, b_kcontig=False, groups=groups, a_sg=k * lda, b_sg=k * ldb,
                                c_sg=m * n, ksegs=segs, a_sk=groups * k * lda, b_sk=groups * k * ldb,
                                rowsum=sums.data_ptr(), rowsum_sg=m, **extra)
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    assert any("ksplit" in nm for nm in names) == (m >= 4), names
    assert rel_err(out, ref) <= TOL[torch.float32]
    if fused:
        assert rel_err(sums, rows) <= TOL[torch.float32]


@pytest.mark.parametrize("k", [512, 640, 767, 898, 1024, 1025, 1283])  # 4 - 11 batches a wave, whole and ragged
@pytest.mark.parametrize("m,n,taken", [(40, 72, True), (512, 1024, True), (513, 1024, False)])
def test_split_contraction_batches(m, n, taken, k):
    """Every remainder of the loop over batches in flight, and both sides of the last tile count that goes here.  Rows and
    columns behind the operands' last hold NaN: nothing of them may reach a result."""
    from rtp_amd import _lib
    gen = torch.Generator().manual_seed(k)
    a, b = _rand((k, m + 3), torch.float32, gen), _rand((k, n + 1), torch.float32, gen)
    a[:, m:], b[:, n:] = float("nan"), float("nan")
    ref = a[:, :m].double().t() @ b[:, :n].double()
    ad, bd = a.to(DEV), b.to(DEV)
    out = torch.full((m, n), float("nan"), device=DEV)
    _lib.profile_enable(1)
    try:
        _ops().gemm_raw(torch.float32, a=ad.data_ptr(), b=bd.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=m + 3,
                        ldb=n + 1, ldc=n, a_kcontig=False, b_kcontig=False)
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    assert any("ksplit" in nm for nm in names) == taken, names
    assert rel_err(out, ref) <= TOL[torch.float32]
