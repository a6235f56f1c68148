"""Two weight gradients in one launch of 256 x 256 tiles (rtp_gemm_pair): bit for bit the two products by themselves, updates and bias
gradients included; pairs that do not fit one round, or that other tiles take, go one after the other."""
import ctypes as C

import pytest
import torch

from test_gpu_gemm import DEV, TOL, rel_err
from test_gpu_gemm_pack import _desc

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _product(gen, m, n, k, groups, shared_a, update):
    """Operands, results and descriptor of `groups` gradients [m, n] over k rows (m and n multiples of 8)."""
    a = torch.randn(k, m if shared_a else groups * m, generator=gen).to(BF).to(DEV)
    b = torch.randn(k, groups * n if shared_a else n, generator=gen).to(BF).to(DEV)
    state = {"grad": torch.full((groups, m * n + 8 * m), float("nan"), dtype=BF, device=DEV)}
    if update:
        state["master"] = torch.randn(groups, m * n + 8 * m, generator=gen).to(DEV)
        state["copy"] = torch.full((groups, m * n + 8 * m), float("nan"), dtype=BF, device=DEV)

    def desc(s):
        kw = dict(a=a.data_ptr(), b=b.data_ptr(), c_out=s["grad"].data_ptr(), m=m, n=n, k=k, lda=a.shape[1], ldb=b.shape[1], ldc=n, groups=groups,
                  a_sg=0 if shared_a else m, b_sg=n if shared_a else 0, c_sg=m * n + 8 * m, a_rowsum=s["grad"].data_ptr() + 2 * m * n,
                  rowsum_sg=m * n + 8 * m)
        if update:
            kw.update(sgd_master=s["master"].data_ptr(), sgd_weights=s["copy"].data_ptr(), sgd_lr=1e-3, sgd_clip=0.05)
        return _desc(**kw)

    ref = torch.stack([(a if shared_a else a[:, g * m:g * m + m]).float().t() @ (b[:, g * n:g * n + n] if shared_a else b).float()
                       for g in range(groups)])
    return state, desc, ref, (m, n)


def _launch(fn):
    from rtp_amd import _lib
    _lib.profile_enable(1)
    try:
        fn(_lib.load(), torch.cuda.current_stream().cuda_stream, _lib.RTP_BF16, _lib.check)
        torch.cuda.synchronize()
        return list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)


@pytest.mark.parametrize("update", [False, True])
@pytest.mark.parametrize("first,second,k,paired", [
    ((2048, 256, 8), (768, 2048, 8), 1024, True),      # an attention layer of width 2048 in 8 shards: 64 + 192 tiles
    ((2048, 512, 4), (1536, 2048, 4), 1504, True),     # ... in 4, a ragged last slab
    ((1536, 1536, 1), (4608, 1536, 1), 2048, True),    # 36 + 108: shares of an XCD that are not whole
    ((1992, 2040, 1), (1304, 2008, 3), 1000, True),    # ragged tiles
    ((2048, 2048, 1), (6400, 2048, 1), 1024, False),   # 64 + 200: more than a round
    ((256, 256, 1), (768, 256, 1), 2048, False)])      # few tiles: other kernels
def test_as_two_launches(first, second, k, paired, update):
    gen = torch.Generator().manual_seed(k)
    one, two = _product(gen, *first[:2], k, first[2], True, update), _product(gen, *second[:2], k, second[2], False, update)
    copies = [{n: t.clone() for n, t in p[0].items()} for p in (one, two)]
    names = _launch(lambda lib, st, dt, check: check(lib.rtp_gemm_pair(st, dt, C.byref(one[1](one[0])), C.byref(two[1](two[0])))))
    if not update or (first[0], k) == (2048, 1024):
        assert ("gemm_bf16_256x256_pair_rc_rc" in names) == paired, names
    _launch(lambda lib, st, dt, check: [check(lib.rtp_gemm(st, dt, C.byref(p[1](s)))) for p, s in zip((one, two), copies)])
    for (state, _, ref, (m, n)), alone in zip((one, two), copies):
        assert rel_err(state["grad"][:, :m * n].reshape(ref.shape), ref) <= TOL[BF]
        for name in state:
            assert torch.equal(state[name][:, :m * n], alone[name][:, :m * n]), name
        assert torch.equal(state["grad"][:, m * n:m * n + m], alone["grad"][:, m * n:m * n + m])  # the row sums
        assert state["grad"][:, m * n + m:].isnan().all()


def test_errors_are_those_of_the_products():
    from rtp_amd import _lib
    gen = torch.Generator().manual_seed(1)
    good, bad = (_product(gen, 2048, 256, 512, 8, True, False) for _ in range(2))
    d, e = good[1](good[0]), bad[1](bad[0])
    e.ldc = 0
    with pytest.raises(_lib.RtpError, match="leading dimensions"):
        _launch(lambda lib, st, dt, check: check(lib.rtp_gemm_pair(st, dt, C.byref(d), C.byref(e))))
    e.ldc, e.m = 256, 0   # an empty product beside a real one
    _launch(lambda lib, st, dt, check: check(lib.rtp_gemm_pair(st, dt, C.byref(d), C.byref(e))))
    assert not good[0]["grad"][:, :2048 * 256].isnan().any() and bad[0]["grad"].isnan().all()


@pytest.mark.parametrize("addend,paired", [("bf16", True), ("fp32", False)])
def test_a_pair_pays_for_the_epilogue_that_the_kernel_finishes_in_a_loop(addend, paired):
    """64 + 64 tiles of ten slabs: together 24 us with an addend in bf16, apart 28; with one in fp32 34 and 28.5."""
    gen = torch.Generator().manual_seed(7)
    m = n = 2048
    k, dt = 640, BF if addend == "bf16" else torch.float32
    descs, held = [], []
    for _ in range(2):
        a, b = (torch.randn(k, r, generator=gen).to(BF).to(DEV) for r in (m, n))
        c, out = torch.randn(m, n, generator=gen).to(dt).to(DEV), torch.full((m, n), float("nan"), dtype=BF, device=DEV)
        held.append((a, b, c, out))
        descs.append(_desc(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=m, ldb=n, ldc=n, c_in=c.data_ptr(), ld_cin=n,
                           flags=0 if addend == "bf16" else 2))
    names = _launch(lambda lib, st, dt, check: check(lib.rtp_gemm_pair(st, dt, C.byref(descs[0]), C.byref(descs[1]))))
    assert ("gemm_bf16_256x256_pair_rc_rc" in names) == paired, names
    for a, b, c, out in held:
        assert rel_err(out, a.float().t() @ b.float() + c.float()) <= TOL[BF]
