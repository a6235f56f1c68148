"""bf16 attention for queries that see no key: hidden by boolean masks (NaN, as nn.MultiheadAttention gives) or pushed down by
large finite ones (which cancel in the softmax), over keys of another sequence and, in the forward pass, its own, against
nn.MultiheadAttention in fp32."""
import pytest
import torch
import torch.nn as nn

from gpu_util import DEV, TOL, rel_err

pytestmark = pytest.mark.gpu

DT = torch.bfloat16


def _pair(E, H, ws):
    from rtp_amd.module.attention import ParallelMultiheadAttention
    ref = nn.MultiheadAttention(E, H).to(DT)
    layer = ParallelMultiheadAttention(E, H, ws, 0, MultiheadAttention_layer=ref, device=DEV, dtype=DT)
    return layer, ref.float()


def _run(layer, ref, L, S, N, E, **masks):
    gen = torch.Generator().manual_seed(L + S)
    q, k, g = (torch.randn(n, N, E, generator=gen).to(DT) for n in (L, S, L))
    qd, kd = (t.to(DEV).requires_grad_() for t in (q, k))
    qf, kf = (t.float().requires_grad_() for t in (q, k))
    out, _ = layer(qd, kd, kd, need_weights=False, **{n: m.to(DEV) for n, m in masks.items()})
    out.backward(g.to(DEV))
    want, _ = ref(qf, kf, kf, need_weights=True, **masks)   # the explicit form: scores + mask, softmax
    want.backward(g.float())
    return [t.detach().float().cpu() for t in (out, qd.grad, kd.grad)], [t.detach() for t in (want, qf.grad, kf.grad)]


@pytest.mark.parametrize("L,S", [(5, 40), (70, 33)])
def test_boolean_masks_that_hide_every_key_give_nan(L, S):
    layer, ref = _pair(128, 4, 2)
    kpm = torch.zeros(3, S, dtype=torch.bool)
    kpm[1] = True
    kpm[2, S // 2:] = True
    got, want = _run(layer, ref, L, S, 3, 128, key_padding_mask=kpm)
    for a, b in zip(got, want):
        assert torch.equal(a[:, 1].isnan(), b[:, 1].isnan()) and b[:, 1].isnan().all()
        assert rel_err(a[:, ::2], b[:, ::2]) <= TOL[DT]
    hidden = torch.zeros(L, S, dtype=torch.bool)
    hidden[L - 1] = True
    got, want = _run(layer, ref, L, S, 3, 128, attn_mask=hidden)
    assert got[0][L - 1].isnan().all() and got[1][L - 1].isnan().all() and got[2].isnan().all() and want[2].isnan().all()
    for a, b in zip(got[:2], want[:2]):
        assert rel_err(a[:L - 1], b[:L - 1]) <= TOL[DT]


@pytest.mark.parametrize("low", [-1e4, -1e9, -1e12, torch.finfo(torch.float32).min])
def test_large_finite_masks_cancel(low):
    layer, ref = _pair(128, 4, 2)
    L, S, N = 40, 70, 3
    bias = torch.zeros(N, S)
    bias[1] = low
    bias[2, S // 2:] = low
    got, want = _run(layer, ref, L, S, N, 128, key_padding_mask=bias)
    for a, b in zip(got, want):
        assert rel_err(a, b) <= TOL[DT]
    mask = torch.randn(L, S, generator=torch.Generator().manual_seed(1))
    mask[7] = low
    got, want = _run(layer, ref, L, S, N, 128, attn_mask=mask)
    for a, b in zip(got, want):
        assert rel_err(a, b) <= TOL[DT]


@pytest.mark.parametrize("low", [-1e4, -1e9, -1e10, -1e12])
def test_large_finite_masks_cancel_in_the_packed_forward(low):
    """Self-attention, running softmax: the maximum is subtracted before the change of base."""
    layer, ref = _pair(128, 4, 2)
    L, N = 70, 3
    x = torch.randn(L, N, 128, generator=torch.Generator().manual_seed(3)).to(DT)
    bias = torch.zeros(N, L)
    bias[1] = low
    bias[2, L // 2:] = low
    mask = torch.randn(L, L, generator=torch.Generator().manual_seed(1))
    mask[7] = low
    for masks in ({"key_padding_mask": bias}, {"attn_mask": mask}):
        with torch.no_grad():
            xd = x.to(DEV)
            out, _ = layer(xd, xd, xd, need_weights=False, **{n: m.to(DEV) for n, m in masks.items()})
            want, _ = ref(x.float(), x.float(), x.float(), need_weights=True, **masks)
        assert rel_err(out, want) <= TOL[DT], list(masks)
