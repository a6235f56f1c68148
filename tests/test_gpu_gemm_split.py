"""fp32 products, whose operands are taken apart into three bf16 numbers: at the edges of tiles, steps of 16 k and slabs of 32, with
segments, groups and row sums, against float64, element by element; and numbers the parts cannot stand for."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu

LAYOUTS = [(True, True), (True, False), (False, True), (False, False)]


def _product(a, b, m, n, k, akc, bkc, ksegs=1, groups=1, rowsum=False):
    """a [ksegs, groups, m, k] and b [ksegs, groups, n, k] in the layouts asked for: product [groups, m, n] and row sums."""
    from rtp_amd import _lib, ops
    # fewer outputs than this would be a kernel for few tiles: copies of the groups, the first of which is looked at
    wanted = groups
    copies = 513 // (-(-m // 32) * -(-n // 32) * groups) + 1
    a, b, groups = a.repeat(1, copies, 1, 1), b.repeat(1, copies, 1, 1), groups * copies
    ad = (a if akc else a.transpose(2, 3)).contiguous().to(DEV)
    bd = (b if bkc else b.transpose(2, 3)).contiguous().to(DEV)
    out = torch.full((groups, m, n), float("nan"), device=DEV)
    sums = torch.full((groups, m), float("nan"), device=DEV)
    _lib.profile_enable(1)
    try:
        done = ops.gemm_raw(torch.float32, a=ad.data_ptr(), b=bd.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k,
                            lda=k if akc else m, ldb=k if bkc else n, ldc=n, a_kcontig=akc, b_kcontig=bkc, groups=groups,
                            a_sg=m * k, b_sg=n * k, c_sg=m * n, ksegs=ksegs, a_sk=groups * m * k, b_sk=groups * n * k,
                            rowsum=sums.data_ptr() if rowsum else None, rowsum_sg=m)
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    # (a row-contiguous operand of fewer than four rows has no vectors: the guarded kernel)
    assert any("_split" in nm for nm in names) or (not akc and m < 4) or (not bkc and n < 4), names
    return out[:wanted].cpu(), sums[:wanted].cpu() if done else None


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(65, 64, 384), (128, 64, 400), (129, 65, 415), (64, 128, 416), (132, 68, 420), (63, 70, 481),
                                   (2, 260, 448), (260, 1, 448), (97, 103, 500), (256, 200, 480)])
@pytest.mark.parametrize("ksegs,groups", [(1, 1), (3, 2)])
def test_edges(akc, bkc, m, n, k, ksegs, groups):
    gen = torch.Generator().manual_seed(m + n + k)
    a, b = torch.randn(ksegs, groups, m, k, generator=gen), torch.randn(ksegs, groups, n, k, generator=gen)
    out, sums = _product(a, b, m, n, k, akc, bkc, ksegs, groups, rowsum=not akc)
    ref = (a.double() @ b.double().transpose(2, 3)).sum(0)
    size = (a.double().abs() @ b.double().abs().transpose(2, 3)).sum(0)
    # parts left out: 3 products of at most 2^-26 of |a| |b|; roundings of the sums: one of 2^-24 per step of 16 k (two for
    # the MFMA's two halves) and one each for the small products, the waves' sums and the result
    steps = ksegs * -(-k // 16)
    assert ((out.double() - ref).abs() <= (3 * 2.0 ** -26 + (2 * steps + 4) * 2.0 ** -24) * size).all()
    if sums is not None:
        rows = a.double().sum((0, 3))
        assert ((sums.double() - rows).abs() <= ksegs * k * 2.0 ** -24 * a.double().abs().sum((0, 3))).all()


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(200, 136, 480), (66, 67, 387)])
def test_numbers_without_parts(akc, bkc, m, n, k):
    """Infinities, NaN, numbers that round to infinity in bf16, overflowing sums: the outputs of the fp32 product, and the
    other rows and columns as if nothing had happened."""
    gen = torch.Generator().manual_seed(m)
    a, b = torch.randn(m, k, generator=gen), torch.randn(n, k, generator=gen)
    a[3, 5], a[m - 1, k - 1], a[40, 0], b[7, 2], b[n - 1, 1] = float("inf"), float("-inf"), float("nan"), float("inf"), 3.4e38
    b[:, 5].clamp_(min=0.5)  # (inf times a number of either sign: infinity or NaN by the order of the sum)
    b[11, 5] = 1.0           # whose second part is zero
    a[50] = 2e38
    out, sums = _product(a[None, None], b[None, None], m, n, k, akc, bkc, rowsum=not akc)
    ref = a.double() @ b.double().t()
    wide = ref.abs() > 3.4028235e38
    plain = ref.isfinite() & ~wide
    size = a.double().abs() @ b.double().abs().t()
    err = (out[0].double() - ref).abs()
    assert (err[plain & (size < 3e38)] <= (k + 4) * 2.0 ** -24 * size[plain & (size < 3e38)]).all()
    assert not out[0][~plain].isfinite().any()
    assert torch.equal(out[0, 3].isnan(), ref[3].isnan()) and (out[0, 3][~ref[3].isnan()] == float("inf")).all()
    assert out[0, 40].isnan().all()
    if sums is not None:
        assert sums[0, 3] == float("inf") and sums[0, 40].isnan() and sums[0, m - 1] == float("-inf")


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
def test_small_numbers(akc, bkc):
    """Operands whose last part has no bits left: the products as precise as those of ordinary numbers."""
    m, n, k = 130, 72, 448
    gen = torch.Generator().manual_seed(1)
    a, b = torch.randn(m, k, generator=gen) * 2.0 ** -118, torch.randn(n, k, generator=gen)
    a[:, ::2] = 0
    out, _ = _product(a[None, None], b[None, None], m, n, k, akc, bkc)
    ref, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    assert ((out[0].double() - ref).abs() <= (k + 4) * 2.0 ** -24 * size + 2.0 ** -149).all()


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("small,large", [(-116, 40), (-119, 40), (-125, 60), (-134, 60), (-140, 80), (-100, -40), (-60, -70),
                                         (100, -30), (110, -60), (60, 30), (-140, 110)])
def test_small_by_large_numbers(akc, bkc, swap, small, large):
    """Operands at 2**small, whose parts would lie below bf16's smallest numbers, by operands at 2**large; and numbers and
    results beyond the range that the parts are scaled to.  As precise as ordinary numbers, subnormal ones included."""
    m, n, k = 130, 72, 448
    gen = torch.Generator().manual_seed(2)
    a, b = torch.randn(m, k, generator=gen) * 2.0 ** small, torch.randn(n, k, generator=gen) * 2.0 ** large
    a[5], b[7] = 0, 0
    if swap:
        a, b, m, n = b, a, n, m
    out, _ = _product(a[None, None], b[None, None], m, n, k, akc, bkc)
    ref, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    steps = -(-k // 16)  # as in test_edges, and half a unit of the smallest subnormal number for the result's rounding
    bound = (3 * 2.0 ** -26 + (2 * steps + 4) * 2.0 ** -24) * size + 2.0 ** -150
    # outputs below fp32's smallest normal number: a sum of products that are subnormal themselves rounds each of them
    bound = torch.where(size < 2.0 ** -126, bound + k * 2.0 ** -150, bound)
    assert ((out[0].double() - ref).abs() <= bound).all()
