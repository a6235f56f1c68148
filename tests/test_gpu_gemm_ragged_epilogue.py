"""The epilogue for results and epilogue operands of any alignment: whole groups of eight columns by 16-byte accesses, a row's last
columns one by one, nothing beside them touched.  Against float64 on the CPU; bf16 results within their rounding (TOL)."""
import pytest
import torch

from test_gpu_gemm import DEV, TOL, rel_err

pytestmark = pytest.mark.gpu
FORMS = ["plain", "bias", "bias a segment", "addend", "fp32 addend", "mask", "bias+addend+mask", "relu", "fp32", "alpha"]


def _shifted(values, shift, pad=3):
    """`values` as rows `pad` elements apart, `shift` elements behind an aligned address; the elements between are NaN."""
    m, n = values.shape
    buf = torch.full((shift + m * (n + pad),), float("nan"), dtype=values.dtype, device=DEV)
    view = buf[shift:].view(m, n + pad)[:, :n]
    view.copy_(values)
    return buf, view


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(65, 67, 320), (130, 1, 520), (129, 255, 64), (700, 521, 72), (2049, 1027, 328)])
@pytest.mark.parametrize("form", FORMS)
def test_forms(dtype, m, n, k, form):
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(m + n)
    segs = 5 if form == "bias a segment" else 1
    a, b = (torch.randn(segs, r, k, generator=gen).to(dtype) for r in (m, n))
    ref = torch.einsum("smk,snk->mn", a.double(), b.double())
    ad, bd = a.to(DEV), b.to(DEV)
    kw, keep = {}, []
    for shift, (what, dt) in enumerate((("addend", torch.float32 if "fp32" in form else dtype), ("mask", dtype)), 1):
        if what not in form:
            continue
        v = torch.randn(m, n, generator=gen).to(dt)
        buf, view = _shifted(v, shift)
        keep.append(buf)
        if what == "addend":
            kw.update(c_in=view.data_ptr(), ld_cin=view.stride(0), cin_f32=dt == torch.float32)
            ref = ref + v.double()
        else:
            kw.update(gate=view.data_ptr(), ld_gate=view.stride(0))
            gate = v
    if "bias" in form:
        bias = torch.randn(segs, n, generator=gen).to(dtype)
        buf, view = _shifted(bias, 1)
        keep.append(buf)
        kw.update(bias=view.data_ptr(), bias_sk=view.stride(0) if segs > 1 else 0)
        ref = ref + bias.double().sum(0)
    if form == "alpha":
        kw["alpha"], ref = 0.25, ref * 0.25
    if form == "relu":
        kw["relu"], ref = True, ref.clamp(min=0)
    if "mask" in form:
        ref = torch.where(gate > 0, ref, torch.zeros_like(ref))
    out_dt = torch.float32 if form == "fp32" else dtype
    buf, out = _shifted(torch.zeros(m, n, dtype=out_dt), 3)
    ops.gemm_raw(dtype, a=ad.data_ptr(), b=bd.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=k, ldb=k, ldc=out.stride(0), a_kcontig=True,
         b_kcontig=True, ksegs=segs, a_sk=m * k, b_sk=n * k, out_f32=out_dt != dtype, **kw)
    assert rel_err(out, ref) <= (TOL[dtype] if out_dt == dtype else 1e-5)
    assert int(torch.isnan(buf).sum()) == buf.numel() - m * n


@pytest.mark.parametrize("pad,shift", [(3, 2), (5, 1)])
@pytest.mark.parametrize("keep", [False, True])
def test_update(pad, shift, keep):
    """Clip + SGD on parameters at odd addresses: bit for bit the separate update of the gradients that the same product leaves."""
    from rtp_amd import ops

    class Sgd:
        lr, clip, keep_grads, missed = 1e-3, 0.05, keep, False
    bf, m, n, k = torch.bfloat16, 136, 264, 328
    gen = torch.Generator().manual_seed(pad)
    a, b = (torch.randn(k, r, generator=gen).to(bf).to(DEV) for r in (m, n))
    bufs = [_shifted(v, shift, pad) for v in (torch.randn(m, n, generator=gen), torch.zeros(m, n, dtype=bf), torch.zeros(m, n, dtype=bf))]
    (_, master), (_, copy), (_, out) = bufs
    old = master.clone()
    kw = dict(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=m, ldb=n, ldc=n + pad, a_kcontig=False,
              b_kcontig=False)
    ops.gemm_raw(bf, sgd=Sgd(), sgd_master=master.data_ptr(), sgd_weights=copy.data_ptr(), **kw)
    assert not Sgd.missed
    if not keep:
        assert not out.any()
        ops.gemm_raw(bf, **kw)
    step = Sgd.lr * out.float().clamp(-Sgd.clip, Sgd.clip)
    assert torch.equal(master, old - step) and torch.equal(copy, (old - step).to(bf))
    for buf, view in bufs:
        assert int(torch.isnan(buf).sum()) == buf.numel() - m * n
