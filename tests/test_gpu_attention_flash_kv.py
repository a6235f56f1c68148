"""rtp_attn_flash_kv_fwd / _bwd: queries and keys of two sequences at the edges of the 32-row groups, the
64- and 128-row workgroups and the key blocks, against float64 on the CPU."""
import pytest
import torch

from gpu_util import DEV, TOL, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,S,d,N,H,G,mask,pad,scale", [
    (1, 1, 32, 1, 1, 1, False, False, 1.0), (31, 33, 64, 2, 2, 1, True, False, 1.0), (33, 31, 128, 1, 2, 2, False, True, 1.0),
    (64, 65, 32, 2, 1, 2, True, True, 1.0), (65, 64, 64, 1, 3, 1, False, False, 1.0), (129, 97, 128, 1, 2, 1, True, True, 1.0),
    (100, 180, 64, 16, 4, 2, False, True, 1.0), (16, 300, 64, 2, 2, 1, False, False, -1.0), (130, 32, 64, 64, 4, 1, True, False, 1.0)])
def test_two_sequences(L, S, d, N, H, G, mask, pad, scale):
    from rtp_amd import ops
    dtype = torch.bfloat16
    gen = torch.Generator().manual_seed(L * 1000 + S)
    e_s, E = H * d, G * H * d
    scale = scale * d ** -0.5
    q, k, v, do = ((torch.randn(n, N, E, generator=gen)).to(dtype) for n in (L, S, S, L))
    m = torch.randn(L, S, generator=gen) if mask else None
    if mask and S > 1:
        m[:, 1::3] = float("-inf")
    kb = None
    if pad:
        kb = torch.zeros(N, S)
        for b in range(N):
            kb[b, S - 1 - b % (S // 2):] = float("-inf")
    ref = [t.double().requires_grad_() for t in (q, k, v)]
    heads = [t.view(t.shape[0], N, G * H, d).permute(1, 2, 0, 3) for t in ref]
    s = heads[0] @ heads[1].transpose(2, 3) * scale
    if m is not None:
        s = s + m.double()
    if kb is not None:
        s = s + kb.double()[:, None, None, :]
    want = (torch.softmax(s, -1) @ heads[2]).permute(2, 0, 1, 3).reshape(L, N, E)
    want.backward(do.double())
    dev = [t.to(DEV) for t in (q, k, v, do)]
    md, kd = (None if t is None else t.to(DEV) for t in (m, kb))
    o, dq = (torch.full_like(dev[0], float("nan")) for _ in range(2))
    dk, dv = (torch.full_like(dev[1], float("nan")) for _ in range(2))
    lse, delta = (torch.empty(G * N * H, L, device=DEV) for _ in range(2))
    st = (N * E, E, d, e_s)
    assert ops.attn_flash_kv_supported(dtype, L, S, d)
    ops.attn_flash_kv_fwd(dev[0], dev[1], dev[2], o, 0, st, st, lse, md, scale, L, S, N, H, d, G, key_bias=kd)
    ops.attn_flash_kv_bwd(dev[0], dev[1], dev[2], o, dev[3], 0, st, st, lse, delta, dq, dk, dv, md, scale, L, S, N, H, d, G,
                          key_bias=kd)
    assert rel_err(o, want) <= TOL[dtype]
    for got, r in zip((dq, dk, dv), ref):
        assert rel_err(got, r.grad) <= TOL[dtype]
