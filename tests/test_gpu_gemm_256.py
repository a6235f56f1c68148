"""The 256 x 256 product kernel's epilogue and row sums where tiles are ragged in both directions (a last tile of 8 rows
and 8 columns), against torch's fp32 product of the same values on the device."""
import pytest
import torch

from test_gpu_gemm import DEV, TOL, _ops, _rand, rel_err

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _run(expect="256x256", **kw):
    from rtp_amd import _lib
    _lib.profile_enable(1)
    try:
        got = _ops().gemm_raw(BF, **kw)
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    assert any(expect in nm for nm in names), names
    return got


def _pair(gen, m, n, k, akc, bkc):
    a = _rand((m, k) if akc else (k, m), BF, gen).to(DEV)
    b = _rand((n, k) if bkc else (k, n), BF, gen).to(DEV)
    return a, b, (a if akc else a.t()).float() @ (b.t() if bkc else b).float()


@pytest.mark.parametrize("akc,bkc,k", [(True, True, 1024), (True, False, 1088), (False, False, 1048), (True, True, 520), (False, False, 512)])
def test_mask_and_row_sums(akc, bkc, k):
    """8 to 17 slabs, whole and ragged last ones: ReLU mask in the epilogue, and the row sums of A beside the product."""
    gen = torch.Generator().manual_seed(k)
    m = n = 3848
    a, b, ref = _pair(gen, m, n, k, akc, bkc)
    gate = _rand((m, n), BF, gen).to(DEV)
    out = torch.full((m, n), float("nan"), dtype=BF, device=DEV)
    sums = torch.full((m,), float("nan"), dtype=BF, device=DEV)
    fused = _run(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(0), ldb=b.stride(0),
                 ldc=n, a_kcontig=akc, b_kcontig=bkc, gate=gate.data_ptr(), ld_gate=n,
                 rowsum=None if akc else sums.data_ptr())
    assert rel_err(out, torch.where(gate.float() > 0, ref, torch.zeros_like(ref))) <= TOL[BF]
    if not akc:
        assert fused and rel_err(sums, a.float().sum(0)) <= TOL[BF]


def test_bias_per_segment_with_fp32_addend_and_output():
    """Two K segments that each carry a bias; addend and output in fp32: 1e-5 covers 1024 fp32 additions per element."""
    gen = torch.Generator().manual_seed(5)
    m = n = 3848
    k, segs = 520, 2
    a = _rand((segs, m, k), BF, gen).to(DEV)
    b = _rand((segs, n, k), BF, gen).to(DEV)
    bias = _rand((segs, n), BF, gen).to(DEV)
    cin = _rand((m, n), torch.float32, gen).to(DEV)
    ref = cin + bias.float().sum(0)
    for s in range(segs):
        ref = ref + a[s].float() @ b[s].float().t()
    out = torch.full((m, n), float("nan"), dtype=torch.float32, device=DEV)
    _run(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=k, ldb=k, ldc=n, a_kcontig=True,
         b_kcontig=True, ksegs=segs, a_sk=m * k, b_sk=n * k, bias=bias.data_ptr(), bias_sk=n, c_in=cin.data_ptr(),
         ld_cin=n, cin_f32=True, out_f32=True)
    assert rel_err(out, ref) <= 1e-5


def test_cross_entropy_gradient_in_the_epilogue():
    """The logits product that turns its tiles into the loss's gradient (2 shards of 1920 classes, a ragged last tile in both
    directions, ignored rows), against the same layer followed by the loss kernels."""
    from rtp_amd import emulate_shards
    from rtp_amd.module.linear import ColumnParallelLinear
    from rtp_amd.module.loss import cross_entropy, linear_cross_entropy
    gen = torch.Generator().manual_seed(3)
    rows, k, vocab = 3848, 1024, 3840
    master = torch.nn.Linear(k, vocab)
    with emulate_shards(2):
        layer = ColumnParallelLinear(k, vocab, linear_layer=master, device=DEV, dtype=BF)
    x = _rand((rows, k), BF, gen).to(DEV)
    target = torch.randint(0, vocab, (rows,), generator=gen)
    target[::7] = -100
    xf, xp = x.clone().requires_grad_(), x.clone().requires_grad_()
    lf = linear_cross_entropy(xf, layer, target.to(DEV))
    lf.backward()
    lp = cross_entropy(layer(xp), target.to(DEV))
    lp.backward()
    assert abs(float(lf.detach()) - float(lp.detach())) <= 1e-6 * abs(float(lp.detach()))
    assert rel_err(xf.grad, xp.grad) <= TOL[BF]
