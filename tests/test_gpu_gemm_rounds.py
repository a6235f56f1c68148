"""bf16 products whose last round of 256 x 256 tiles would be mostly idle, or whose last row of tiles mostly padding, run as two
launches over their rows: every operand that has rows moves along, values as of one launch."""
import pytest
import torch

from test_gpu_gemm import DEV, TOL, rel_err
from test_gpu_gemm_256 import _pair

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _names(fn):
    from rtp_amd import _lib
    _lib.profile_enable(1)
    try:
        fn()
        torch.cuda.synchronize()
        return {n: s["launches"] if isinstance(s, dict) else s for n, s in dict(_lib.profile_collect()).items()}
    finally:
        _lib.profile_enable(0)


SHAPES = [(4352, 4096, 1544), (4360, 4104, 1032), (2312, 8192, 1032), (1032, 16384, 520)]  # 256, 520, 264 and 8 rows behind the cut
UPDATED = [(4352, 4096, 4096), (8200, 4096, 2048), (6144, 3072, 4096)]  # an update is cut where the K loop is long enough
FORMS = ["plain", "bias", "addend", "fp32 addend", "mask", "fp32"]


@pytest.mark.parametrize("akc,bkc,form,m,n,k",
                         [(True, bkc, form, *shape) for bkc in (True, False) for form in FORMS for shape in SHAPES] +
                         [(False, False, form, *shape) for form in ("plain", "addend", "row sums", "accumulated") for shape in SHAPES] +
                         [(False, False, "update", *shape) for shape in UPDATED])
def test_forms(akc, bkc, m, n, k, form):
    """Weight gradients (the last layout) with row sums, added to earlier ones and both, and with an update."""
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(m + k)
    a, b, ref = _pair(gen, m, n, k, akc, bkc)
    kw, dt = {}, BF
    sums = torch.full((m,), float("nan"), dtype=BF, device=DEV)
    out = torch.full((m, n), float("nan"), dtype=torch.float32 if form == "fp32" else BF, device=DEV)
    if "addend" in form:
        c = torch.randn(m, n, generator=gen).to(torch.float32 if "fp32" in form else BF).to(DEV)
        kw, ref = dict(c_in=c.data_ptr(), ld_cin=n, cin_f32="fp32" in form), ref + c.float()
    elif form == "accumulated":  # gradients on top of what is there, the bias's too
        out.copy_(torch.randn(m, n, generator=gen))
        sums.copy_(torch.randn(m, generator=gen))
        ref, old_sums = ref + out.float(), sums.float()
        kw = dict(c_in=out.data_ptr(), ld_cin=n, rowsum=sums.data_ptr(), rowsum_accum=True)
    elif form == "bias":
        bias = torch.randn(n, generator=gen).to(BF).to(DEV)
        kw, ref = dict(bias=bias.data_ptr()), ref + bias.float()
    elif form == "mask":
        gate = torch.randn(m, n, generator=gen).to(BF).to(DEV)
        kw, ref = dict(gate=gate.data_ptr(), ld_gate=n), torch.where(gate > 0, ref, torch.zeros_like(ref))
    elif form == "fp32":
        kw, dt = dict(out_f32=True), torch.float32
    elif form == "row sums":
        kw = dict(rowsum=sums.data_ptr())
    elif form == "update":
        class Sgd:
            lr, clip, keep_grads, missed = 1e-3, 0.05, True, False
        master = torch.randn(m, n, generator=gen).to(DEV)
        old, copy = master.clone(), torch.full((m, n), float("nan"), dtype=BF, device=DEV)
        kw = dict(sgd=Sgd(), sgd_master=master.data_ptr(), sgd_weights=copy.data_ptr())
    names = _names(lambda: ops.gemm_raw(BF, a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(0),
                                        ldb=b.stride(0), ldc=n, a_kcontig=akc, b_kcontig=bkc, **kw))
    assert len(names) == 2 and any("256x256" in name for name in names), names
    assert rel_err(out, ref) <= (TOL[BF] if dt == BF else 1e-5)
    assert not out.isnan().any()
    if form == "row sums":
        assert rel_err(sums, a.float().sum(0)) <= TOL[BF]
    if form == "accumulated":
        assert rel_err(sums, a.float().sum(0) + old_sums) <= TOL[BF]
    if form == "update":
        step = Sgd.lr * out.float().clamp(-Sgd.clip, Sgd.clip)
        assert torch.equal(master, old - step) and torch.equal(copy, (old - step).to(BF))


@pytest.mark.parametrize("m,n,groups,two", [(4352, 4096, 1, True), (4096, 4096, 1, False), (1100, 1024, 16, True)])
def test_route_and_groups(m, n, groups, two):
    """Where two launches are taken, and groups whose rows are cut alike, against each group's product in fp32."""
    from rtp_amd import ops
    k = 1024
    gen = torch.Generator().manual_seed(groups)
    a, b = (torch.randn(groups, r, k, generator=gen).to(BF).to(DEV) for r in (m, n))
    out = torch.full((groups, m, n), float("nan"), dtype=BF, device=DEV)
    names = _names(lambda: ops.gemm_raw(BF, a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=k, ldb=k, ldc=n,
                                        a_kcontig=True, b_kcontig=True, groups=groups, a_sg=m * k, b_sg=n * k, c_sg=m * n))
    assert (len(names) == 2) == two, names
    for g in range(groups):
        assert rel_err(out[g], a[g].float() @ b[g].float().t()) <= TOL[BF]


@pytest.mark.parametrize("akc,bkc,update", [(True, True, False), (True, False, False), (False, False, False), (False, False, True)])
@pytest.mark.parametrize("m,extra", [(4128, 32), (8200, 8)])
def test_equal_rows_are_equal_on_either_side_of_the_cut(akc, bkc, update, m, extra):
    """The few rows behind the cut are by themselves a product that gemm_kwaves.hip would take, whose sums have another order.  Equal bits, row sums
    and updated parameters too; an update of 4128 rows is not cut, so it goes over 8200 alone."""
    from rtp_amd import ops
    if update and m != 8200:
        m, extra = 8224, 32
    n, k = 4096, 2048
    gen = torch.Generator().manual_seed(m)
    a, b, ref = _pair(gen, m, n, k, akc, bkc)
    rows = a if akc else a.t()
    rows[m - extra:] = rows[:extra]
    ref[m - extra:] = ref[:extra]
    out, sums = torch.full((m, n), float("nan"), dtype=BF, device=DEV), torch.full((m,), float("nan"), dtype=BF, device=DEV)
    kw, compared = {}, [out]
    if not akc:
        kw["rowsum"] = sums.data_ptr()
        compared.append(sums)
    if update:
        class Sgd:
            lr, clip, keep_grads, missed = 1e-3, 0.05, True, False
        master = torch.randn(m, n, generator=gen).to(DEV)
        master[m - extra:] = master[:extra]
        copy = torch.full((m, n), float("nan"), dtype=BF, device=DEV)
        kw.update(sgd=Sgd(), sgd_master=master.data_ptr(), sgd_weights=copy.data_ptr())
        compared += [master, copy]
    names = _names(lambda: ops.gemm_raw(BF, a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(0),
                                        ldb=b.stride(0), ldc=n, a_kcontig=akc, b_kcontig=bkc, **kw))
    assert len(names) == 2, names
    assert rel_err(out, ref) <= TOL[BF] and not out.isnan().any()
    for t in compared:
        assert torch.equal(t[m - extra:], t[:extra])
