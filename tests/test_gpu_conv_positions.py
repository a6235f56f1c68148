"""The convolution's input gradient where a slab is one kernel position of 32 channels: channel counts that fill whole slabs,
all but a quarter of them and just too little, shards whose channels end inside a slab, strides that skip pixels, dilation, 32- and 64-row
tiles, channels-last gradients and a run in the middle of a wider one, against torch's input gradient in fp64 on the CPU."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,ci,h,w,co,shards,k,s,p,d", [
    (2, 3, 9, 11, 32, 1, (3, 3), (1, 1), (0, 0), (1, 1)), (1, 33, 7, 8, 24, 3, (3, 2), (1, 1), (1, 2), (1, 2)),
    (3, 70, 6, 6, 48, 4, (1, 1), (1, 1), (0, 0), (1, 1)), (2, 32, 13, 12, 20, 2, (5, 3), (2, 1), (2, 1), (1, 1)),
    (1, 65, 17, 16, 40, 8, (3, 3), (3, 2), (1, 0), (2, 1)), (2, 8, 10, 10, 66, 3, (3, 3), (1, 1), (1, 1), (1, 1)),
    (1, 1, 5, 5, 160, 5, (5, 5), (1, 1), (2, 2), (1, 1)),
    # 33 to 64 rows by positions in both types, the last slab not full; 5 x 5 weights that are read as they lie, and a few tiles of them
    (3, 70, 6, 6, 72, 4, (1, 1), (1, 1), (0, 0), (1, 1)), (2, 40, 9, 9, 29, 1, (3, 3), (1, 1), (1, 1), (1, 1)),
    (1, 65, 17, 16, 48, 8, (3, 3), (3, 2), (1, 0), (2, 1)), (1, 64, 9, 9, 32, 2, (5, 5), (1, 1), (2, 2), (1, 1)),
    (2, 16, 8, 8, 30, 3, (5, 5), (1, 1), (2, 2), (1, 1)), (1, 40, 12, 12, 64, 4, (2, 2), (1, 1), (0, 0), (1, 1))])
def test_input_gradient_against_torch(n, ci, h, w, co, shards, k, s, p, d, dtype):
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(co + h)
    g = ops.conv_geom((n, ci, h, w), k, s, p, d)
    kp, n_s, extra = ci * k[0] * k[1], co // shards, 5
    flat = torch.randn(shards, extra + n_s * kp + n_s, generator=gen).to(dtype)
    flat[:, :extra], flat[:, extra + n_s * kp:] = float("nan"), float("nan")  # around the weights: nothing of it comes through
    dy = torch.randn(n, co + 2, g.ho, g.wo, generator=gen).to(dtype)
    dy[:, 0], dy[:, -1] = float("nan"), float("nan")
    weight = torch.cat([r[extra:extra + n_s * kp].view(n_s, ci, *k) for r in flat]).double()
    grad = dy[:, 1:-1].double()
    want = torch.nn.grad.conv2d_input((n, ci, h, w), weight, grad, s, p, d)
    terms = torch.nn.grad.conv2d_input((n, ci, h, w), weight.abs(), grad.abs(), s, p, d)
    # products of bf16 are exact in fp32: a sum of K terms in any order is within K units of 2^-24 of their magnitudes, and the
    # result rounds once more (bf16 has 8 significant bits: half a unit of the last one is at most 2^-8 of the value)
    bound = terms * (co * k[0] * k[1] + 1) * 2.0 ** -24 + want.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 0)
    for fmt in (torch.contiguous_format, torch.channels_last):
        dx = torch.empty(n, ci, h, w, dtype=dtype, device=DEV)
        ops.conv2d_dgrad(dy.to(DEV).contiguous(memory_format=fmt), g, flat.to(DEV), extra, n_s, 1, dx)
        assert bool(((dx.cpu().double() - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,ci,h,co,shards,k,s,p", [
    (1, 3, 6, 32, 1, 3, 1, 0), (7, 5, 10, 40, 2, 3, 1, 0), (3, 33, 8, 64, 4, 1, 1, 0), (5, 4, 17, 30, 3, 3, 2, 1),
    (2, 16, 6, 130, 5, 3, 1, 1), (9, 2, 4, 72, 1, 1, 1, 0)])
def test_weight_gradient_of_whole_runs(n, ci, h, co, shards, k, s, p, dtype):
    """Planes of output pixels that runs of four or eight divide are read by runs, others and channels-last gradients by elements: the
    same sums in the same order, so the same bits; images of 16 - 100 pixels end inside slabs of 32."""
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(co + h)
    g = ops.conv_geom((n, ci, h, h), (k, k), (s, s), (p, p), (1, 1))
    kp, n_s = ci * k * k, co // shards
    x = torch.randn(n, ci, h, h, generator=gen).to(dtype)
    dy = torch.randn(n, co + 2, g.ho, g.wo, generator=gen).to(dtype)
    dy[:, 0], dy[:, -1] = float("nan"), float("nan")
    got = []
    for fmt in (torch.contiguous_format, torch.channels_last):
        grads = torch.zeros(shards, n_s * (kp + 1), dtype=dtype, device=DEV)
        ops.conv2d_wgrad(dy.to(DEV).contiguous(memory_format=fmt), x.to(DEV), g, grads, 0, n_s * kp, n_s, 1, False)
        got.append(grads.cpu())
    assert torch.equal(got[0], got[1])
    shape, d64, x64 = (co, ci, k, k), dy[:, 1:-1].double(), x.double()
    weight, bias = torch.nn.grad.conv2d_weight(x64, shape, d64, s, p), d64.sum((0, 2, 3))
    w_abs, b_abs = torch.nn.grad.conv2d_weight(x64.abs(), shape, d64.abs(), s, p), d64.abs().sum((0, 2, 3))
    rows = got[0].double()
    for have, want, terms in ((rows[:, :n_s * kp].reshape(shape), weight, w_abs), (rows[:, n_s * kp:].reshape(co), bias, b_abs)):
        bound = terms * (n * g.ho * g.wo + 1) * 2.0 ** -24 + want.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 0)
        assert bool(((have - want).abs() <= bound).all())


@pytest.mark.parametrize("n,h,ci,co,p", [(1, 129, 40, 70, 1), (9, 61, 100, 32, 0), (3, 75, 64, 24, 1), (2, 129, 40, 70, 1), (6, 75, 64, 24, 1),
                                         (6, 75, 33, 22, 0)])
def test_input_gradient_of_many_bf16_pixels(n, h, ci, co, p):
    """More tiles of 64 x 64 than CUs or twice as many, some taken as 64 x 128: ragged last ones, 40 to 100 rows, contractions of whole positions and of mixed slabs,
    against fp64 on the CPU; inputs of few bits make every sum exact in fp32, so that only the rounding to bf16 is left."""
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(co)
    g = ops.conv_geom((n, ci, h, h), (3, 3), (1, 1), (p, p), (1, 1))
    dy = torch.randint(-3, 4, (n, co, g.ho, g.wo), generator=gen).to(torch.bfloat16)
    flat = torch.randint(-3, 4, (2, co // 2 * ci * 9), generator=gen).to(torch.bfloat16)
    dx = torch.empty(n, ci, h, h, dtype=torch.bfloat16, device=DEV)
    ops.conv2d_dgrad(dy.to(DEV), g, flat.to(DEV), 0, co // 2, 0, dx)
    want = torch.nn.grad.conv2d_input((n, ci, h, h), flat.view(co, ci, 3, 3).double(), dy.double(), 1, p)
    assert torch.equal(dx.cpu(), want.to(torch.bfloat16))
