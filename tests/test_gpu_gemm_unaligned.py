"""rtp_gemm where addresses, leading dimensions or extents are no multiples of 16 bytes: the register-staged loaders and
the element-wise epilogue, at the edges of tiles, vectors and K slabs, against float64 on the CPU."""
import pytest
import torch

from gpu_util import DEV, TOL, rel_err

pytestmark = pytest.mark.gpu


def _unaligned(shape, ld, dtype, gen):
    """The values on the CPU and a device copy that starts one element into its allocation, rows `ld` apart, the gaps NaN."""
    host = (torch.randn(shape, generator=gen) * 0.5).to(dtype)
    buf = torch.full((1 + shape[0] * ld,), float("nan"), dtype=dtype, device=DEV)
    view = buf[1:].view(shape[0], ld)[:, :shape[1]]
    view.copy_(host)
    return host, view


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("akc,bkc", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("m,n,k", [(65, 67, 8), (63, 129, 9), (129, 71, 63), (127, 257, 65), (70, 1001, 129), (9, 8, 515),
                                   (2050, 2051, 67)])
def test_layouts(dtype, akc, bkc, m, n, k):
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(m + n + k)
    a, ad = _unaligned((m, k) if akc else (k, m), (k if akc else m) + 1, dtype, gen)
    b, bd = _unaligned((n, k) if bkc else (k, n), (k if bkc else n) + 3, dtype, gen)
    bias, biasd = _unaligned((1, n), n, dtype, gen)
    gate, gated = _unaligned((m, n), n, dtype, gen)
    cin, cind = _unaligned((m, n), n + 1, dtype, gen)
    A, B = (a if akc else a.t()).double(), (b if bkc else b.t()).double()
    ref = (A @ B.t() + bias.double() + cin.double()) * (gate > 0)
    buf = torch.full((1 + m * (n + 2),), -7.0, dtype=dtype, device=DEV)
    out = buf[1:].view(m, n + 2)
    sums = torch.full((m,), -7.0, dtype=dtype, device=DEV)
    fused = ops.gemm_raw(dtype, a=ad.data_ptr(), b=bd.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=ad.stride(0),
                         ldb=bd.stride(0), ldc=n + 2, a_kcontig=akc, b_kcontig=bkc, bias=biasd.data_ptr(),
                         gate=gated.data_ptr(), ld_gate=n, c_in=cind.data_ptr(), ld_cin=n + 1, rowsum=sums.data_ptr())
    assert fused == (not akc)
    assert rel_err(out[:, :n], ref) <= TOL[dtype]
    assert torch.equal(out[:, n:], torch.full_like(out[:, n:], -7.0)) and buf[0] == -7.0
    if fused:
        assert rel_err(sums, A.sum(1)) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [33, 128, 131])
def test_k_segments(dtype, k):
    """A row-parallel layer of odd width: the weight's K runs in segments that lie an odd distance apart."""
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(k)
    m, n, segs = 150, 99, 3
    x, xd = _unaligned((m, segs * k), segs * k, dtype, gen)
    w, wd = _unaligned((segs, n * k), n * k + 1, dtype, gen)
    ref = sum(x[:, s * k:(s + 1) * k].double() @ w[s].view(n, k).double().t() for s in range(segs))
    out = torch.full((m, n), float("nan"), dtype=dtype, device=DEV)
    ops.gemm_raw(dtype, a=xd.data_ptr(), b=wd.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=segs * k, ldb=k, ldc=n,
                 a_kcontig=True, b_kcontig=True, ksegs=segs, a_sk=k, b_sk=n * k + 1)
    assert rel_err(out, ref) <= TOL[dtype]
