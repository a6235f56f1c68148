"""The 256 x 256 product kernel where a workgroup goes through several tiles: its loads run on into the next tile while the epilogue of
the last one is written, so every form of the epilogue, K segment ends, ragged last slabs and ragged tiles are met between two tiles.
Against torch's fp32 product of the same values on the device; bf16 results within their rounding (TOL), fp32 ones within 1e-5, which
covers some hundred fp32 additions an element."""
import pytest
import torch

from test_gpu_gemm import DEV, TOL, _ops, _rand, rel_err
from test_gpu_gemm_256 import _pair, _run

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# 17 x 17 and 33 x 17 tiles, ragged in both directions: no split over the XCDs; 16 x 24: bricks.  The first two are cut at most contractions, and
# their last rows go to other tiles (test_gpu_gemm_rounds.py); ONE_LAUNCH are not: 27 x 16 ragged in both directions, 33 x 15 in rows.
ONE_LAUNCH = [(4096, 6144), (6664, 3872), (8200, 3840)]
SHAPES = [(4344, 4264), (8200, 4344)] + ONE_LAUNCH


def _run_alone(shape, **kw):
    """The product; of the shapes of ONE_LAUNCH it is one kernel's, more tiles than CUs."""
    from rtp_amd import _lib
    _lib.profile_enable(1)
    try:
        got = _ops().gemm_raw(BF, **kw)
        torch.cuda.synchronize()
        launches = {name: s["launches"] for name, s in _lib.profile_collect().items()}
    finally:
        _lib.profile_enable(0)
    if shape in ONE_LAUNCH:
        assert list(launches.values()) == [1] and "256x256" in next(iter(launches)), launches
    return got


@pytest.mark.parametrize("akc,bkc", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("k", [136, 192, 264])
def test_plain(akc, bkc, m, n, k):
    """Three slabs with a ragged last one, three whole ones, five with a ragged one."""
    gen = torch.Generator().manual_seed(m + k)
    a, b, ref = _pair(gen, m, n, k, akc, bkc)
    out = torch.full((m, n), float("nan"), dtype=BF, device=DEV)
    _run_alone((m, n), a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(0), ldb=b.stride(0), ldc=n,
               a_kcontig=akc, b_kcontig=bkc)
    assert rel_err(out, ref) <= TOL[BF]


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("form", ["bias", "bias+relu", "relu", "addend", "mask", "mask+addend", "bias+addend", "alpha", "stream",
                                  "fp32", "fp32 addend", "row sums"])
def test_epilogues(m, n, form):
    gen = torch.Generator().manual_seed(n)
    k = 520
    akc = form != "row sums"
    a, b, ref = _pair(gen, m, n, k, akc, akc)
    kw, dt = {}, BF
    if form == "alpha":
        kw["alpha"], ref = 0.125, ref * 0.125
    if "addend" in form:
        c = _rand((m, n), torch.float32 if "fp32" in form else BF, gen).to(DEV)
        kw.update(c_in=c.data_ptr(), ld_cin=n, cin_f32="fp32" in form)
        ref = ref + c.float()
    if "bias" in form:
        bias = _rand((n,), BF, gen).to(DEV)
        kw["bias"], ref = bias.data_ptr(), ref + bias.float()
    if "relu" in form:
        kw["relu"], ref = True, ref.clamp(min=0)
    if "mask" in form:
        gate = _rand((m, n), BF, gen).to(DEV)
        gate[::3, ::5] = 0.0
        gate[1::7, 3::11] = float("nan")
        kw.update(gate=gate.data_ptr(), ld_gate=n)
        ref = torch.where(gate.float() > 0, ref, torch.zeros_like(ref))
    if form == "stream":
        kw["stream_out"] = True
    if form == "fp32":
        kw["out_f32"], dt = True, torch.float32
    sums = torch.full((m,), float("nan"), dtype=BF, device=DEV)
    if form == "row sums":
        kw["rowsum"] = sums.data_ptr()
    out = torch.full((m, n), float("nan"), dtype=dt, device=DEV)
    done = _run_alone((m, n), a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(0), ldb=b.stride(0), ldc=n,
                      a_kcontig=akc, b_kcontig=akc, **kw)
    assert rel_err(out, ref) <= (TOL[BF] if dt == BF else 1e-5)
    if form == "row sums":
        assert done and rel_err(sums, a.float().sum(0)) <= TOL[BF]


@pytest.mark.parametrize("form", ["plain", "bias", "bias+relu", "addend", "mask", "stream", "in place"])
@pytest.mark.parametrize("m,n,groups", [(6664, 3872, 1), (2766, 384, 8), (4100, 264, 6), (3000, 1000, 3)])
def test_ragged_tiles_touch_their_own_alone(m, n, groups, form):
    """Waves of a ragged tile that lie inside, across an edge and outside: results in the midst of NaN, addends, masks and biases too, whose
    surroundings stay as they are and out of the sums."""
    gen = torch.Generator().manual_seed(m + n)
    k, gap = 200, 24
    a = _rand((m, k), BF, gen).to(DEV)
    b = _rand((groups, n, k), BF, gen).to(DEV)
    ref = torch.stack([a.float() @ w.float().t() for w in b])

    def field(rows, value=None):  # [groups, rows, n] whose rows, and groups, lie `gap` elements or more apart
        whole = torch.full((groups, rows + 2, n + gap), float("nan"), dtype=BF, device=DEV)
        if value is not None:
            whole[:, 1:rows + 1, :n] = value
        return whole, whole[:, 1:rows + 1, :n]

    whole, out = field(m)
    kw = {}
    if form.startswith("bias"):
        _, bias = field(1, _rand((groups, 1, n), BF, gen).to(DEV))
        kw, ref = dict(bias=bias.data_ptr(), bias_sg=bias.stride(0), relu="relu" in form), ref + bias.float()
        ref = ref.clamp(min=0) if "relu" in form else ref
    elif form == "addend":
        _, c = field(m, _rand((groups, m, n), BF, gen).to(DEV))
        kw, ref = dict(c_in=c.data_ptr(), ld_cin=c.stride(1), cin_sg=c.stride(0)), ref + c.float()
    elif form == "in place":
        out.copy_(_rand((groups, m, n), BF, gen))
        kw, ref = dict(c_in=out.data_ptr(), ld_cin=out.stride(1), cin_sg=out.stride(0)), ref + out.float()
    elif form == "mask":
        _, gate = field(m, _rand((groups, m, n), BF, gen).to(DEV))
        kw = dict(gate=gate.data_ptr(), ld_gate=gate.stride(1), gate_sg=gate.stride(0))
        ref = torch.where(gate.float() > 0, ref, torch.zeros_like(ref))
    elif form == "stream":
        kw = dict(stream_out=True)
    _run(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=k, ldb=k, ldc=out.stride(1), a_kcontig=True,
         b_kcontig=True, groups=groups, b_sg=n * k, c_sg=out.stride(0), **kw)
    assert rel_err(out, ref) <= TOL[BF] and not out.isnan().any()
    out.fill_(float("nan"))
    assert whole.isnan().all()


@pytest.mark.parametrize("segs,k", [(2, 72), (3, 64), (17, 64)])
def test_segments_and_their_biases(segs, k):
    """K segments that end inside a tile, of one slab and of two with a ragged one; a bias a segment (17: more than a wave's page holds)."""
    gen = torch.Generator().manual_seed(segs)
    m, n = 4096, 6144
    a = _rand((segs, m, k), BF, gen).to(DEV)
    b = _rand((segs, n, k), BF, gen).to(DEV)
    bias = _rand((segs, n), BF, gen).to(DEV)
    ref = bias.float().sum(0) + sum(a[s].float() @ b[s].float().t() for s in range(segs))
    out = torch.full((m, n), float("nan"), dtype=BF, device=DEV)
    _run(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=k, ldb=k, ldc=n, a_kcontig=True,
         b_kcontig=True, ksegs=segs, a_sk=m * k, b_sk=n * k, bias=bias.data_ptr(), bias_sk=n)
    assert rel_err(out, ref) <= TOL[BF]


@pytest.mark.parametrize("groups", [3, 8])
def test_groups(groups):
    """Tiles of several groups, with and without a split over the XCDs, a bias a group."""
    gen = torch.Generator().manual_seed(groups)
    m, n, k = 2056, 4104, 264
    a = _rand((groups, m, k), BF, gen).to(DEV)
    b = _rand((groups, k, n), BF, gen).to(DEV)
    bias = _rand((groups, n), BF, gen).to(DEV)
    out = torch.full((groups, m, n), float("nan"), dtype=BF, device=DEV)
    _run(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=k, ldb=n, ldc=n, a_kcontig=True, b_kcontig=False,
         groups=groups, a_sg=m * k, b_sg=k * n, c_sg=m * n, bias=bias.data_ptr(), bias_sg=n)
    for g in range(groups):
        assert rel_err(out[g], a[g].float() @ b[g].float() + bias[g].float()) <= TOL[BF], g


def test_values_beyond_the_contraction_do_not_count():
    """What lies behind a row's last k in memory, and in the LDS from slabs before, may be anything."""
    gen = torch.Generator().manual_seed(9)
    m, n, k, ld = 6664, 3872, 136, 192
    a = torch.full((m, ld), float("nan"), dtype=BF, device=DEV)
    b = torch.full((n, ld), float("inf"), dtype=BF, device=DEV)
    a[:, :k] = _rand((m, k), BF, gen).to(DEV)
    b[:, :k] = _rand((n, k), BF, gen).to(DEV)
    out = torch.full((m, n), float("nan"), dtype=BF, device=DEV)
    _run_alone((m, n), a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=ld, ldb=ld, ldc=n, a_kcontig=True, b_kcontig=True)
    assert rel_err(out, a[:, :k].float() @ b[:, :k].float().t()) <= TOL[BF]


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("n,groups", [(248, 8), (256, 12), (456, 8), (512, 8), (520, 8), (768, 6), (776, 6), (1032, 4), (4104, 1)])
def test_row_sums_over_the_tile_columns(n, groups, accumulate):
    """One to four tile columns and more, which share the sums of a tile's rows among them: the bits of the smaller tiles, each row once."""
    gen = torch.Generator().manual_seed(n)
    m, k = 4104, 264
    a, b = _rand((k, groups * m), BF, gen).to(DEV), _rand((k, n), BF, gen).to(DEV)
    old = _rand((groups, m), BF, gen).to(DEV) if accumulate else torch.full((groups, m), float("nan"), dtype=BF, device=DEV)
    results = []
    for cols, run in ((n, _run), (64, _ops().gemm_raw)):
        sums = old.clone()
        out = torch.full((groups, m, cols), float("nan"), dtype=BF, device=DEV)
        kw = dict(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=cols, k=k, lda=groups * m, ldb=n, ldc=cols, a_kcontig=False,
                  b_kcontig=False, groups=groups, a_sg=m, c_sg=m * cols, rowsum=sums.data_ptr(), rowsum_sg=m, rowsum_accum=accumulate)
        assert run(**kw) if run is _run else run(BF, **kw)
        results.append(sums)
    ref = a.float().sum(0).view(groups, m) + (old.float() if accumulate else 0)
    assert rel_err(results[0], ref) <= TOL[BF] and torch.equal(*results)


@pytest.mark.parametrize("m,n,k", [(6144, 2048, 200), (4096, 4096, 136), (4104, 3808, 264),    # 192, 256 and 255 tiles
                                   (4096, 6144, 520), (6664, 3872, 136), (6664, 3872, 520), (8200, 3840, 264)])  # 384, 432, 495
@pytest.mark.parametrize("keep,clip", [(False, 0.05), (True, 0.0)])
def test_update(m, n, k, keep, clip):
    """Clip + SGD on a tile's parameters, several tiles a workgroup, ragged ones too: bit for bit the separate update of the gradients that the
    same product leaves (which the kernel writes where they are kept)."""
    class Sgd:
        lr, keep_grads, missed = 1e-3, keep, False
    Sgd.clip = clip
    gen = torch.Generator().manual_seed(m + n)
    a, b, ref = _pair(gen, m, n, k, False, False)
    master = _rand((m, n), torch.float32, gen).to(DEV)
    old, copy = master.clone(), torch.full((m, n), float("nan"), dtype=BF, device=DEV)
    out = torch.full((m, n), float("nan"), dtype=BF, device=DEV)
    kw = dict(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=m, ldb=n, ldc=n, a_kcontig=False, b_kcontig=False)
    _run_alone((m, n), sgd=Sgd(), sgd_master=master.data_ptr(), sgd_weights=copy.data_ptr(), stream_out=True, **kw)
    if keep:
        assert rel_err(out, ref) <= TOL[BF]
        grad = out.clone()
    else:
        assert out.isnan().all()
        _run_alone((m, n), **kw)
        grad = out
    g32 = grad.float()
    if clip:
        g32 = g32.clamp(-clip, clip)
    step = Sgd.lr * g32
    assert torch.equal(master, old - step)
    assert torch.equal(copy, (old - step).to(BF))


@pytest.mark.parametrize("shift,gap,large", [(0, 32, True), (0, 8, False), (8, 32, False)])
def test_updates_of_parameters_that_are_no_whole_lines_go_elsewhere(shift, gap, large):
    """Groups of parameters at a multiple of 128 bytes or not: the tiles differ, the results do not."""
    from rtp_amd import _lib

    class Sgd:
        lr, clip, keep_grads, missed = 1e-3, 0.05, True, False

    gen = torch.Generator().manual_seed(shift + gap)
    m, n, k, groups = 1024, 2048, 264, 8
    a, b = _rand((k, groups * m), BF, gen).to(DEV), _rand((k, n), BF, gen).to(DEV)
    step = m * n + gap
    master = _rand((shift + groups * step,), torch.float32, gen).to(DEV)[shift:].view(groups, step)
    old, copy, out = master.clone(), *(torch.full((shift + groups * step,), float("nan"), dtype=BF, device=DEV)[shift:].view(groups, step) for _ in range(2))
    _lib.profile_enable(1)
    try:
        _ops().gemm_raw(BF, a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=groups * m, ldb=n, ldc=n, a_kcontig=False,
                        b_kcontig=False, groups=groups, a_sg=m, c_sg=step, sgd=Sgd(), sgd_master=master.data_ptr(), sgd_weights=copy.data_ptr())
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    assert any("256x256" in name for name in names) == large, names
    grad, rest = out[:, :m * n], slice(m * n, None)
    assert rel_err(grad.reshape(groups, m, n), torch.stack([a[:, g * m:g * m + m].float().t() @ b.float() for g in range(groups)])) <= TOL[BF]
    new = old[:, :m * n] - Sgd.lr * grad.float().clamp(-Sgd.clip, Sgd.clip)
    assert torch.equal(master[:, :m * n], new) and torch.equal(copy[:, :m * n], new.to(BF))
    assert torch.equal(master[:, rest], old[:, rest]) and copy[:, rest].isnan().all() and out[:, rest].isnan().all()


@pytest.mark.parametrize("m,n,k", [(2048, 4096, 1024), (2040, 4096, 1000), (1288, 4608, 1032)])
def test_row_sums_shared_by_two_wave_columns(m, n, k):
    """The 256 x 128 tile, whose wave columns sum two of a wave tile's four row blocks each: every row once, whole and ragged tiles, on top of what is
    there and alone.  A sum of k terms in fp32 is within k units of 2^-24 of their magnitudes, and rounds to bf16's 8 bits (half a unit: 2^-8)."""
    gen = torch.Generator().manual_seed(k)
    a, b = _rand((k, m), BF, gen).to(DEV), _rand((k, n), BF, gen).to(DEV)
    old = _rand((m,), BF, gen).to(DEV)
    out = torch.empty(m, n, dtype=BF, device=DEV)
    for accumulate in (False, True):
        sums = old.clone()
        fused = _run("256x128", a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=m, ldb=n, ldc=n, a_kcontig=False,
                     b_kcontig=False, rowsum=sums.data_ptr(), rowsum_accum=accumulate)
        want = a.double().sum(0) + (old.double() if accumulate else 0)
        bound = (k + 2) * 2.0 ** -24 * (a.double().abs().sum(0) + old.double().abs()) + 2.0 ** -8 * want.abs()
        assert fused and bool(((sums.double() - want).abs() <= bound).all())
    assert rel_err(out, a.float().t() @ b.float()) <= TOL[BF]
