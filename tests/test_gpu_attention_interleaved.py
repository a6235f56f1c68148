"""The running-softmax attention core's backward over blocks of 64 rows without edges (whose vector work runs between the MFMAs) beside
blocks with edges, and its results' stores by whole lines, against float64 on the CPU: one block, ragged ends, the causal diagonal at every
wave of a workgroup, hidden keys, results inside wider rows."""
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
