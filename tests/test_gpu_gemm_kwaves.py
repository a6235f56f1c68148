"""Products with few output tiles and a long contraction, the contraction split over the waves of a workgroup: against float64 in
every layout, at contractions that leave waves without slabs, with a ragged last slab or a ragged round of slabs in flight, over K
segments and groups, with every addend and mask of the epilogue and with row sums."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu

LAYOUTS = [(True, True), (True, False), (False, True), (False, False)]


def _run(dtype, a, b, m, n, k, akc, bkc, *, taken=True, **kw):
    from rtp_amd import _lib, ops
    _lib.profile_enable(1)
    try:
        done = ops.gemm_raw(dtype, a=a.data_ptr(), b=b.data_ptr(), m=m, n=n, k=k, a_kcontig=akc, b_kcontig=bkc, **kw)
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    assert any("kwaves" in nm for nm in names) == taken, names
    return done


def _bound(dtype, steps, size, ref):
    """One rounding of 2^-24 per MFMA (two halves), of the eight waves' sums and of the epilogue; the result's own rounding."""
    return (2 * steps + 12) * 2.0 ** -24 * size + (2.0 ** -8 * ref.abs() if dtype == torch.bfloat16 else 0.0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
# aligned; aligned but for the output; odd (with slabs and rounds of slabs that end anywhere)
@pytest.mark.parametrize("m,n,k", [(8, 64, 512), (32, 32, 520), (40, 24, 1024), (64, 256, 1032), (136, 72, 2056), (8, 8, 4104),
                                   (24, 1000, 776), (36, 68, 520), (40, 12, 2048), (33, 65, 513), (9, 31, 1027), (70, 101, 2055),
                                   (31, 8, 4099)])
@pytest.mark.parametrize("ksegs,groups", [(1, 1), (3, 2)])
def test_edges(dtype, akc, bkc, m, n, k, ksegs, groups, taken=True):
    pad = 8 if k % 8 == 0 else 7
    if dtype == torch.float32 and not akc and not bkc and pad == 7:
        pytest.skip("unaligned row-contiguous fp32 operands have a kernel of their own")
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(ksegs, groups, m, k, generator=gen).to(dtype)
    b = torch.randn(ksegs, groups, n, k, generator=gen).to(dtype)
    # NaN behind the last row and column of each matrix: nothing of it may reach a result
    A = torch.full((ksegs, groups, m, k + pad) if akc else (ksegs, groups, k, m + pad), float("nan"), dtype=dtype)
    B = torch.full((ksegs, groups, n, k + pad) if bkc else (ksegs, groups, k, n + pad), float("nan"), dtype=dtype)
    A[..., :k if akc else m] = a if akc else a.transpose(2, 3)
    B[..., :k if bkc else n] = b if bkc else b.transpose(2, 3)
    A, B = A.to(DEV), B.to(DEV)
    out = torch.full((groups, m, n), float("nan"), dtype=dtype, device=DEV)
    sums = torch.full((groups, m), float("nan"), dtype=dtype, device=DEV)
    done = _run(dtype, A, B, m, n, k, akc, bkc, taken=taken, c_out=out.data_ptr(), lda=A.stride(2), ldb=B.stride(2), ldc=n, groups=groups,
                a_sg=A.stride(1), b_sg=B.stride(1), c_sg=m * n, ksegs=ksegs, a_sk=A.stride(0), b_sk=B.stride(0),
                rowsum=None if akc else sums.data_ptr(), rowsum_sg=m)
    ref = (a.double() @ b.double().transpose(2, 3)).sum(0)
    size = (a.double().abs() @ b.double().abs().transpose(2, 3)).sum(0)
    steps = ksegs * -(-k // (16 if dtype == torch.bfloat16 else 2))
    assert ((out.cpu().double() - ref).abs() <= _bound(dtype, steps, size, ref)).all()
    if done:
        rows, size = a.double().sum((0, 3)), a.double().abs().sum((0, 3))
        assert ((sums.cpu().double() - rows).abs() <= _bound(dtype, ksegs * k, size, rows)).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
# more than 256 tiles of 32 x 32 and at most 256 of 64 x 32: whole and ragged, the last 64 rows all there, half or a sliver
@pytest.mark.parametrize("m,n,k", [(192, 1408, 2048), (264, 1032, 2056), (72, 2728, 2112), (100, 2101, 2051), (65, 2753, 2049)])
def test_taller_tiles(dtype, akc, bkc, m, n, k):
    test_edges(dtype, akc, bkc, m, n, k, 1, 1, taken=dtype == torch.float32 or akc == bkc)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("akc,bkc", [(True, True), (True, False)])
def test_epilogue(dtype, akc, bkc):
    m, n, k = 40, 96, 1040
    gen = torch.Generator().manual_seed(3)
    a, b = (torch.randn(m, k, generator=gen).to(dtype).to(DEV), torch.randn(n, k, generator=gen).to(dtype).to(DEV))
    bt = b if bkc else b.t().contiguous()
    bias, gate = torch.randn(n, generator=gen).to(dtype).to(DEV), torch.randn(m, n, generator=gen).to(dtype).to(DEV)
    cin = torch.randn(m, n, generator=gen).to(DEV)
    prod = (a.double() @ b.double().t()).cpu()
    size = (a.double().abs() @ b.double().abs().t()).cpu() + 16
    common = dict(lda=k, ldb=k if bkc else n, ldc=n)
    for f32 in (True, False):
        for relu in (False, True):  # (a ReLU's sums keep their order)
            out = torch.empty(m, n, dtype=torch.float32 if f32 else dtype, device=DEV)
            _run(dtype, a, bt, m, n, k, akc, bkc, taken=not relu, c_out=out.data_ptr(), bias=bias.data_ptr(),
                 c_in=cin.data_ptr(), ld_cin=n, cin_f32=True, out_f32=f32, relu=relu, **common)
            ref = prod + bias.double().cpu() + cin.double().cpu()
            ref = ref.clamp(min=0) if relu else ref
            assert ((out.cpu().double() - ref).abs() <= _bound(out.dtype, k // 2, size, ref)).all()
    out = torch.empty(m, n, dtype=dtype, device=DEV)
    _run(dtype, a, bt, m, n, k, akc, bkc, c_out=out.data_ptr(), gate=gate.data_ptr(), ld_gate=n, alpha=0.5, **common)
    ref = 0.5 * prod * (gate.cpu() > 0)
    assert ((out.cpu().double() - ref).abs() <= _bound(dtype, k // 2, size, ref)).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_update_is_that_of_the_plain_gradient(dtype):
    """clip + SGD in the epilogue: bit for bit the update by the gradient that the product without it stores."""
    from rtp_amd import ops
    m, n, k = 72, 136, 700
    gen = torch.Generator().manual_seed(2)
    a, b = (torch.randn(k, c, generator=gen).to(dtype).to(DEV) for c in (m, n))
    w = torch.randn(m, n, generator=gen).to(DEV)
    grad, kept, master, copy = (torch.zeros(m, n, dtype=t, device=DEV) for t in (dtype, dtype, torch.float32, dtype))
    master.copy_(w)
    common = dict(lda=m, ldb=n, ldc=n)
    _run(dtype, a, b, m, n, k, False, False, c_out=grad.data_ptr(), **common)
    sgd = ops.FusedSgd(lr=0.1, clip=20.0, keep_grads=True)
    _run(dtype, a, b, m, n, k, False, False, c_out=kept.data_ptr(), sgd=sgd, sgd_master=master.data_ptr(),
         sgd_weights=copy.data_ptr() if dtype == torch.bfloat16 else 0, **common)
    assert not sgd.missed and torch.equal(kept, grad) and float(grad.abs().max()) > 20.0
    assert torch.equal(master, w - 0.1 * grad.float().clamp(-20.0, 20.0))
    if dtype == torch.bfloat16:
        assert torch.equal(copy, master.to(dtype))
