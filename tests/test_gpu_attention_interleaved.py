"""The running-softmax attention core's backward over blocks of 64 rows without edges (whose vector work runs between the MFMAs) beside
blocks with edges, and its results' stores by whole lines, against float64 on the CPU: one block, ragged ends, hidden keys, results inside wider
rows in workgroups of two waves; the causal diagonal at every wave of a workgroup of four, with and without a key bias, and masks, which have
kernels without the interleaved loop, element by element."""
import pytest
import torch

from gpu_util import DEV, TOL, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("L,causal,pad", [(64, False, False), (65, True, True), (127, False, True), (128, True, False), (193, True, False),
                                          (255, False, False), (320, True, True)])
def test_packed_self_attention(L, causal, pad, d):
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(L * 8 + d)
    N, H, G = 2, 2, 1
    e_s, E = H * d, H * d
    ld = 3 * E + 8 * d  # rows with a gap behind q, k and v, which stays as it is
    qkv = torch.randn(L, N, ld, generator=gen).to(torch.bfloat16)
    do = torch.randn(L, N, E, generator=gen).to(torch.bfloat16)
    kb = None
    if pad:
        kb = torch.zeros(N, L)
        kb[1, L - 40:] = float("-inf")
    ref = [qkv[:, :, i * E:(i + 1) * E].double().requires_grad_() for i in range(3)]
    q, k, v = (t.view(L, N, H, d).permute(1, 2, 0, 3) for t in ref)
    s = q @ k.transpose(2, 3) * d ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(L, L).triu(1).bool(), float("-inf"))
    if kb is not None:
        s = s + kb.double()[:, None, None, :]
    want = (torch.softmax(s, -1) @ v).permute(2, 0, 1, 3).reshape(L, N, E)
    want.backward(do.double())
    xd, dd, kd = qkv.to(DEV), do.to(DEV), None if kb is None else kb.to(DEV)
    o = torch.full_like(dd, float("nan"))
    dx = torch.full_like(xd, 7.0)
    lse, delta = (torch.empty(G * N * H, L, device=DEV) for _ in range(2))
    st, os_ = (N * ld, ld, d, 3 * e_s), (N * E, E, d, e_s)
    ops.attn_flash_fwd(xd, 0, E, 2 * E, st, o, 0, os_, lse, None, causal, d ** -0.5, L, N, H, d, G, key_bias=kd)
    ops.attn_flash_bwd(xd, 0, E, 2 * E, st, o, dd, 0, os_, lse, delta, dx, None, causal, d ** -0.5, L, N, H, d, G, key_bias=kd)
    assert rel_err(o, want) <= TOL[torch.bfloat16]
    for i, r in enumerate(ref):
        assert rel_err(dx[:, :, i * E:(i + 1) * E], r.grad) <= TOL[torch.bfloat16]
    assert torch.equal(dx[:, :, 3 * E:], torch.full_like(dx[:, :, 3 * E:], 7.0))


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("L,N,H,form", [(193, 16, 8, "causal"), (193, 16, 8, "causal, key bias"), (193, 16, 8, "key bias"), (256, 16, 8, "causal"),
                                        (193, 16, 8, "mask"), (130, 1, 3, "mask"), (64, 2, 2, "mask"), (33, 5, 3, "causal")])
def test_every_element(L, N, H, form, d):
    """Workgroups of four waves from 256 of them on (128 heads of 129 rows or more), of two below."""
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(L + d)
    E = H * d
    qkv, do = (torch.randn(L, N, n * E, generator=gen).to(torch.bfloat16) for n in (3, 1))
    add, kb, mask = torch.zeros(N, 1, L, L, dtype=torch.float64), None, None
    if "causal" in form:
        add = add.masked_fill(torch.ones(L, L).triu(1).bool(), float("-inf"))
    if "key bias" in form:  # hidden keys at the end, but never all of a query's
        kb = torch.randn(N, L, generator=gen)
        kb[1::2, L - 70:] = float("-inf")
        add = add + kb.double()[:, None, None, :]
    if form == "mask":
        mask = torch.randn(L, L, generator=gen)
        mask[torch.rand(L, L, generator=gen) < 0.3] = float("-inf")
        mask[:, 0] = 0.0
        add = add + mask.double()
    heads = lambda t: t.double().view(L, N, H, d).permute(1, 2, 0, 3)
    back = lambda t: t.permute(2, 0, 1, 3).reshape(L, N, E)
    (q, k, v), g, c = (heads(t) for t in qkv.chunk(3, -1)), heads(do), d ** -0.5
    p = torch.softmax(q @ k.transpose(2, 3) * c + add, -1)
    out = p @ v
    delta = (g * out).sum(-1, keepdim=True)
    ds = p * (g @ v.transpose(2, 3) - delta)
    # bf16 keeps 8 significant bits: half a unit of the last one is at most u = 2^-8 of the value.  P and dS are rounded once, as factors; O once, and
    # delta is formed from it; results once.  The fp32 sums of up to 256 terms and the exponentials of scores below 16 are within 2^-16 of their
    # terms: a sixteenth of u covers them.
    u = 2.0 ** -8
    near = u + u / 16
    ds_err = near * (ds.abs() + p * (g.abs() * out.abs()).sum(-1, keepdim=True)) + u / 16 * p * (g.abs() @ v.abs().transpose(2, 3))
    wants = [(ds @ k * c, ds_err @ k.abs() * c), (ds.transpose(2, 3) @ q * c, ds_err.transpose(2, 3) @ q.abs() * c),
             (p.transpose(2, 3) @ g, near * (p.transpose(2, 3) @ g.abs()))]
    xd, dd = qkv.to(DEV), do.to(DEV)
    kd, md = (None if t is None else t.to(DEV) for t in (kb, mask))
    o, dx = torch.empty_like(dd), torch.empty_like(xd)
    lse, delta_d = (torch.empty(N * H, L, device=DEV) for _ in range(2))
    st, os_ = (3 * N * E, 3 * E, d, 3 * E), (N * E, E, d, E)
    ops.attn_flash_fwd(xd, 0, E, 2 * E, st, o, 0, os_, lse, md, "causal" in form, c, L, N, H, d, 1, key_bias=kd)
    ops.attn_flash_bwd(xd, 0, E, 2 * E, st, o, dd, 0, os_, lse, delta_d, dx, md, "causal" in form, c, L, N, H, d, 1, key_bias=kd)
    wants.append((out, near * (p @ v.abs())))
    for got, (want, err) in zip(list(dx.cpu().chunk(3, -1)) + [o.cpu()], wants):
        bound = err + u * (want.abs() + err)
        assert bool(((got.double() - back(want)).abs() <= back(bound)).all())


@pytest.mark.parametrize("L,N,H,d", [(32, 1, 1, 64), (5, 3, 3, 64), (32, 257, 8, 64), (31, 2049, 1, 64), (32, 5, 1, 32), (9, 7, 1, 128)])
def test_short_sequences_store_their_rows_alone(L, N, H, d):
    """The short-sequence core with one, two and four problems a workgroup, the last of them not full: results of every problem,
    and nothing beside them."""
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(L * 8 + d)
    E, gap = H * d, 8
    ld = 3 * E + gap
    qkv = torch.randn(L, N, ld, generator=gen).to(torch.bfloat16)
    do = torch.randn(L, N, E, generator=gen).to(torch.bfloat16)
    ref = [qkv[:, :, i * E:(i + 1) * E].double().requires_grad_() for i in range(3)]
    q, k, v = (t.view(L, N, H, d).permute(1, 2, 0, 3) for t in ref)
    want = (torch.softmax(q @ k.transpose(2, 3) * d ** -0.5, -1) @ v).permute(2, 0, 1, 3).reshape(L, N, E)
    want.backward(do.double())
    xd, dd = qkv.to(DEV), do.to(DEV)
    o, dx = torch.full((L, N, E + gap), 7.0, dtype=torch.bfloat16, device=DEV), torch.full_like(xd, 7.0)
    p = torch.empty(N * H, L, L, dtype=torch.bfloat16, device=DEV)
    st = (N * ld, ld, d, 3 * E)
    ops.attn_fwd(xd, 0, E, 2 * E, st, o, 0, (N * (E + gap), E + gap, d, E), p, None, False, d ** -0.5, L, N, H, d, 1)
    ops.attn_bwd(xd, 0, E, 2 * E, st, dd, 0, (N * E, E, d, E), p, dx, d ** -0.5, L, N, H, d, 1)
    assert rel_err(o[:, :, :E], want) <= TOL[torch.bfloat16]
    for i, r in enumerate(ref):
        assert rel_err(dx[:, :, i * E:(i + 1) * E], r.grad) <= TOL[torch.bfloat16]
    assert torch.equal(o[:, :, E:], torch.full_like(o[:, :, E:], 7.0))
    assert torch.equal(dx[:, :, 3 * E:], torch.full_like(dx[:, :, 3 * E:], 7.0))
