"""Large bf16 products on operands that are not vector-aligned run on aligned copies where the caller offers scratch memory (the Python
side does): bit for bit the product that reads its operands where they are (called without scratch memory), in every layout."""
import ctypes as C

import pytest
import torch

from test_gpu_gemm import DEV, TOL, rel_err

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
ALLOC = C.CFUNCTYPE(C.c_void_p, C.c_void_p, C.c_size_t)


def _desc(**kw):
    from rtp_amd import _lib
    d = _lib.GemmDesc()
    d.batch = d.zdiv = d.groups = d.ksegs = 1
    d.alpha = 1.0
    for name, v in kw.items():
        setattr(d, name, v)
    return d


def _direct(kw, alloc=None):
    """rtp_gemm without the Python side's scratch memory."""
    from rtp_amd import _lib
    lib = _lib.load()
    names = {"rowsum": "a_rowsum"}
    flags = 4 if kw.get("relu") else 0
    d = _desc(**{names.get(k, k): v for k, v in kw.items() if k not in ("relu",)})
    d.flags = flags
    if alloc is not None:
        assert lib.rtp_gemm_workspace(alloc, None) == 0
    try:
        _lib.check(lib.rtp_gemm(torch.cuda.current_stream().cuda_stream, _lib.RTP_BF16, C.byref(d)))
    finally:
        if alloc is not None:
            lib.rtp_gemm_workspace(None, None)
    torch.cuda.synchronize()


def _packed(kw, expect=True):
    from rtp_amd import _lib, ops
    _lib.profile_enable(1)
    try:
        ops.gemm_raw(BF, **kw)
        torch.cuda.synchronize()
        names = list(_lib.profile_collect())
    finally:
        _lib.profile_enable(0)
    assert ("gemm_pack" in names) == expect, names
    return names


def _operand(gen, rows, k, kc, copies, gap, shift):
    """`copies` matrices [rows, k] stored k- or row-contiguous, NaN between their lines and around them."""
    lines, length = (rows, k) if kc else (k, rows)
    buf = torch.full((shift + copies * lines * (length + gap) + 16,), float("nan"), dtype=BF, device=DEV)
    view = buf[shift:shift + copies * lines * (length + gap)].view(copies, lines, length + gap)[:, :, :length]
    view.copy_(torch.randn(copies, lines, length, generator=gen).to(BF))
    return buf, view, (view if kc else view.transpose(1, 2))


LAYOUTS = [  # k-contiguous a / b, m, n, k, groups, segments, (gap between lines, shift of the first) of a / b; (0, 0): vector-aligned
    (True, True, 4097, 2056, 1032, 1, 2, (0, 0), (2, 3)), (True, True, 4100, 2051, 520, 4, 1, (0, 0), (1, 0)),
    (True, False, 4097, 4104, 1023, 1, 2, (0, 0), (1, 1)), (False, True, 4097, 4104, 1023, 1, 2, (3, 2), (0, 0)),
    (False, False, 1027, 4099, 777, 3, 4, (0, 5), (1, 1)), (True, False, 1027, 4099, 777, 3, 4, (2, 7), (0, 0)),
    (True, False, 4097, 4096, 1023, 1, 1, (1, 1), (0, 0)), (False, False, 4099, 4096, 500, 1, 1, (5, 1), (0, 0)),
    (False, False, 5000, 4096, 2050, 1, 1, (0, 0), (1, 2)), (False, True, 4097, 2056, 1032, 1, 2, (0, 1), (0, 0))]


@pytest.mark.parametrize("akc,bkc,m,n,k,groups,segs,place_a,place_b", LAYOUTS)
def test_layouts(akc, bkc, m, n, k, groups, segs, place_a, place_b):
    gen = torch.Generator().manual_seed(m + n + k)
    abuf, a, af = _operand(gen, m, k, akc, groups * segs, *place_a)
    bbuf, b, bf = _operand(gen, n, k, bkc, segs, *place_b)   # shared by the groups
    ref = sum(af.view(groups, segs, m, k)[:, s].float() @ bf[s].float().t() for s in range(segs))
    outs = []
    for run in (_packed, _direct):
        out = torch.full((groups, m, n), float("nan"), dtype=BF, device=DEV)
        run(dict(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(1), ldb=b.stride(1), ldc=n,
                 a_kcontig=akc, b_kcontig=bkc, groups=groups, ksegs=segs, a_sg=segs * a.stride(0), a_sk=a.stride(0), b_sk=b.stride(0),
                 c_sg=m * n))
        outs.append(out)
    assert rel_err(outs[0], ref) <= TOL[BF]
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("form", ["bias+relu", "addend", "mask", "row sums"])
@pytest.mark.parametrize("n", [2304, 2301])
def test_epilogues(form, n):
    gen = torch.Generator().manual_seed(n)
    m, k, akc = 4098, 3000, form != "row sums"
    _, a, af = _operand(gen, m, k, akc, 1, *((0, 0) if akc else (1, 1)))
    _, b, bf = _operand(gen, n, k, akc, 1, 1, 1)
    extra = torch.randn(m, n, generator=gen).to(BF).to(DEV)
    kw = {"bias+relu": dict(bias=extra.data_ptr(), relu=True), "addend": dict(c_in=extra.data_ptr(), ld_cin=n),
          "mask": dict(gate=extra.data_ptr(), ld_gate=n), "row sums": {}}[form]
    outs = []
    for run in (_packed, _direct):
        out = torch.full((m, n), float("nan"), dtype=BF, device=DEV)
        sums = torch.full((m,), float("nan"), dtype=BF, device=DEV)
        if form == "row sums":
            kw = dict(rowsum=sums.data_ptr())
        run(dict(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(1), ldb=b.stride(1), ldc=n,
                 a_kcontig=akc, b_kcontig=akc, **kw))
        outs.append((out, sums))
    assert torch.equal(outs[0][0], outs[1][0])
    if form == "row sums":
        assert rel_err(outs[0][1], af[0].float().sum(1)) <= TOL[BF] and torch.equal(outs[0][1], outs[1][1])


def test_non_finite_values_stay_in_their_rows():
    gen = torch.Generator().manual_seed(1)
    m, n, k = 4098, 4096, 1501
    _, a, af = _operand(gen, m, k, True, 1, 1, 1)
    _, b, bf = _operand(gen, n, k, False, 1, 0, 0)
    a[0, 17, k - 1], a[0, m - 1, 0] = float("nan"), float("inf")
    outs = []
    for run in (_packed, _direct):
        out = torch.zeros(m, n, dtype=BF, device=DEV)
        run(dict(a=a.data_ptr(), b=b.data_ptr(), c_out=out.data_ptr(), m=m, n=n, k=k, lda=a.stride(1), ldb=b.stride(1), ldc=n,
                 a_kcontig=True, b_kcontig=False))
        outs.append(out)
    bad = ~torch.isfinite(outs[0]).all(1)
    assert bad.nonzero().flatten().tolist() == [17, m - 1]
    assert torch.equal(torch.nan_to_num(outs[0]), torch.nan_to_num(outs[1])) and torch.equal(outs[0].isnan(), outs[1].isnan())


def test_without_memory_and_small_products_go_the_old_way():
    gen = torch.Generator().manual_seed(2)
    for (m, n, k), expect in (((4098, 4096, 2050), True), ((300, 301, 300), False)):
        _, a, _ = _operand(gen, m, k, False, 1, 1, 1)
        _, b, _ = _operand(gen, n, k, False, 1, 0, 0)
        out, refused = (torch.zeros(m, n, dtype=BF, device=DEV) for _ in range(2))
        kw = dict(a=a.data_ptr(), b=b.data_ptr(), m=m, n=n, k=k, lda=a.stride(1), ldb=b.stride(1), ldc=n, a_kcontig=False, b_kcontig=False)
        _packed(dict(kw, c_out=out.data_ptr()), expect)
        asked = []
        no = ALLOC(lambda ctx, size: asked.append(size))
        _direct(dict(kw, c_out=refused.data_ptr()), no)
        assert bool(asked) == expect and torch.equal(out, refused)


def test_captured_layer_and_two_streams():
    """A column layer of odd shards: the scratch memory of a captured step belongs to its graph, that of an eager one to its stream."""
    from rtp_amd import emulate_shards
    from rtp_amd.module.linear import ColumnParallelLinear
    torch.manual_seed(0)
    with emulate_shards(4):
        layer = ColumnParallelLinear(4096, 4 * 501, device=DEV, dtype=BF)
    xs = [torch.randn(4100, 4096, device=DEV).to(BF) for _ in range(3)]
    dy = torch.randn(4100, 4 * 501, device=DEV).to(BF)

    def step(x):
        x = x.detach().requires_grad_()
        layer.zero_grad()
        y = layer(x)
        y.backward(dy)
        return [y.detach(), x.grad] + [p.grad.clone() for p in layer.parameters()]

    from rtp_amd import _lib
    _lib.profile_enable(1)
    try:
        want = [step(x) for x in xs]
        torch.cuda.synchronize()
        assert "gemm_pack" in _lib.profile_collect()
    finally:
        _lib.profile_enable(0)
    static = xs[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            got = step(static)
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(got, want[0]))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = step(static)
    for i in (1, 2, 0, 1):
        static.copy_(xs[i])
        graph.replay()
        eager = step(xs[(i + 1) % 3])
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(held, want[i]))
        assert all(torch.equal(a, b) for a, b in zip(eager, want[(i + 1) % 3]))


# weight gradients of 100, 256 (64 x 32), 160 and 232 tiles, an input gradient of 88; the last one's 512 x 600 are 304 tiles of 32 x 32
@pytest.mark.parametrize("akc,bkc,m,n,k,few", [(False, False, 300, 300, 8192, True), (False, False, 500, 1000, 8000, True),
                                               (False, False, 130, 1000, 8190, True), (False, False, 500, 900, 8000, True),
                                               (True, False, 250, 333, 9001, True), (True, False, 512, 600, 12001, False)])
def test_few_tiles_stay_with_their_kernel(akc, bkc, m, n, k, few):
    """What gemm_kwaves.hip takes it takes at any alignment, scratch memory or not: its order of the sums is another one."""
    gen = torch.Generator().manual_seed(m + n + k)
    _, a, af = _operand(gen, m, k, akc, 1, 1, 1)
    _, b, bf = _operand(gen, n, k, bkc, 1, 1, 1)
    outs = [torch.full((m, n), float("nan"), dtype=BF, device=DEV) for _ in range(2)]
    kw = dict(a=a.data_ptr(), b=b.data_ptr(), m=m, n=n, k=k, lda=a.stride(1), ldb=b.stride(1), ldc=n, a_kcontig=akc, b_kcontig=bkc)
    names = _packed(dict(kw, c_out=outs[0].data_ptr()), not few)
    assert not few or (len(names) == 1 and "kwaves" in names[0]), names
    _direct(dict(kw, c_out=outs[1].data_ptr()))
    assert torch.equal(*outs)
    assert rel_err(outs[0], af[0].float() @ bf[0].float().t()) <= TOL[BF]


def test_a_refusal_of_memory_is_remembered():
    """Where torch's allocator has no memory left it is asked once and not by every product; a second later it is asked again."""
    import time

    from rtp_amd import ops
    gen = torch.Generator().manual_seed(3)
    m, n, k = 4098, 4096, 2050
    _, a, _ = _operand(gen, m, k, False, 1, 1, 1)
    _, b, _ = _operand(gen, n, k, False, 1, 1, 1)
    outs = [torch.zeros(m, n, dtype=BF, device=DEV) for _ in range(7)]
    kw = dict(a=a.data_ptr(), b=b.data_ptr(), m=m, n=n, k=k, lda=a.stride(1), ldb=b.stride(1), ldc=n, a_kcontig=False, b_kcontig=False)
    refusals = lambda: torch.cuda.memory_stats()["num_ooms"]  # noqa: E731
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total, fill = torch.cuda.get_device_properties(DEV).total_memory, []
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (4 << 20)) / total)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):  # what the allocator still holds in pieces
            while True:
                fill.append(torch.empty(8 << 20, dtype=torch.uint8, device=DEV))
        before = refusals()
        for out in outs[:5]:
            ops.gemm_raw(BF, c_out=out.data_ptr(), **kw)
        assert refusals() == before + 1
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        fill.clear()
        time.sleep(1.1)
    _packed(dict(kw, c_out=outs[5].data_ptr()))
    _direct(dict(kw, c_out=outs[6].data_ptr()))
    assert all(torch.equal(out, outs[6]) for out in outs[:6])
