"""rtp_gemm_warm_next on products of few and of many slabs: a wave asks for the hinted region a few KiB a slab, and neither a
region that leaves most waves without a piece nor one beyond what a launch can take changes a bit of the result."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 192, 320, 1000, 2048])
@pytest.mark.parametrize("warm_bytes", [5 * 1024, (3 << 20) + 16, 80 << 20])
def test_hint_over_the_slabs(k, warm_bytes):
    from rtp_amd import _lib, ops
    lib = _lib.load()
    gen = torch.Generator().manual_seed(k)
    dtype, m, n = torch.bfloat16, 1024, 2048
    a, w = (torch.randn(r, k, generator=gen).to(dtype).to(DEV) for r in (m, n))
    res = torch.randn(m, n, generator=gen).to(dtype).to(DEV)
    region = torch.ones(warm_bytes, dtype=torch.uint8, device=DEV)

    def product(hint):
        out = torch.full((m, n), float("nan"), dtype=dtype, device=DEV)
        if hint:
            _lib.check(lib.rtp_gemm_warm_next(region.data_ptr(), warm_bytes))
        ops.gemm_raw(dtype, a=a.data_ptr(), b=w.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=k, ldb=k, ldc=n, a_kcontig=True,
                     b_kcontig=True, c_in=res.data_ptr(), ld_cin=n)
        return out

    plain, hinted = product(False), product(True)
    assert lib.rtp_gemm_warm_pending() == 0
    torch.cuda.synchronize()
    assert torch.equal(plain, hinted)
    assert bool((region == 1).all())
    want = res.double().cpu() + a.double().cpu() @ w.double().cpu().t()
    assert float((plain.double().cpu() - want).norm() / want.norm()) <= 2 ** -8  # one rounding to bf16, and fp32 sums
