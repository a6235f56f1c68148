"""The softmax of attention scores and its backward over rows that fill a lane's registers to the last, by one more, and that are too
long for them, with every addend, against float64."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("l,s", [(3, 1), (7, 63), (5, 64), (9, 65), (4, 256), (6, 257), (3, 512), (2, 513), (5, 1024), (3, 1025), (2, 2048),
                                 (3, 2049), (70, 70), (90, 33)])
@pytest.mark.parametrize("form", ["plain", "causal", "mask", "masks", "bias", "keep"])
def test_rows(dtype, l, s, form):
    from rtp_amd import ops
    n, heads, groups = 2, 3, 2
    z = groups * n * heads
    gen = torch.Generator().manual_seed(l * 1000 + s)
    scores, scale = torch.randn(z, l, s, generator=gen) * 4, 0.37
    kw, add = dict(mask=None, causal=form == "causal"), torch.zeros(z, l, s, dtype=torch.float64)
    if form == "causal":
        add = torch.full((l, s), float("-inf"), dtype=torch.float64).triu(s - l + 1).expand(z, l, s)
    if form in ("mask", "masks"):
        m = torch.randn((l, s) if form == "mask" else (4, l, s), generator=gen)
        m = torch.where(torch.rand(m.shape, generator=gen) < 0.2, torch.tensor(float("-inf")), m)
        m[..., 0] = 0.5  # (every query sees a key)
        kw["mask"] = m.to(DEV)
        add = m.double().expand(z, l, s) if form == "mask" else m.double().repeat(z // 4, 1, 1)
    if form == "bias":
        b = torch.randn(n, s, generator=gen)
        kw.update(key_bias=b.to(DEV), heads=heads)
        add = b.double()[(torch.arange(z) // heads) % n][:, None, :].expand(z, l, s)
    p = torch.full((z, l, s), 7.0, dtype=dtype, device=DEV)
    keep = None
    if form == "keep":
        keep = ((torch.rand(z, l, s, generator=gen) < 0.8) / 0.8).float()
        kw.update(keep=keep.to(DEV), p_dropped=torch.full_like(p, 7.0))
    ops.softmax_fwd(scores.to(DEV), p, scale=scale, **kw)
    ref = torch.softmax(scores.double() * scale + add, -1)
    if form == "causal" and l > s:
        ref[:, :l - s] = 0  # queries before the first key: no probability anywhere
    own = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    # the exponent's argument, of up to 2^5, is rounded three times; exp, the sum of s / 64 + 6 terms and two more operations
    bound = (3 * 2.0 ** 5 + s / 64 + 12) * 2.0 ** -24
    assert ((p.cpu().double() - ref).abs() <= (bound + own) * ref + 1e-37).all()
    if keep is not None:
        assert torch.equal(kw["p_dropped"].cpu(), (p.cpu().float() * keep).to(dtype))
    dp, ds = torch.randn(z, l, s, generator=gen), torch.full_like(p, 7.0)
    ops.softmax_bwd(p, dp.to(DEV), ds, scale, keep=None if keep is None else keep.to(DEV))
    pd, g = p.cpu().double(), dp.double() if keep is None else dp.double() * keep.double()
    want = scale * pd * (g - (pd * g).sum(-1, keepdim=True))
    size = scale * pd * (g.abs() + (pd * g.abs()).sum(-1, keepdim=True))
    assert ((ds.cpu().double() - want).abs() <= (s / 64 + 12) * 2.0 ** -24 * size + own * want.abs() + 1e-37).all()
