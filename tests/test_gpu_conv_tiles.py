"""The convolution's tile kernel at its edges -- row counts around the 32- and 64-row tiles, contractions that end inside
a slab, one element of everything, strides and padding, several shards in one tile, split contractions of the weight
gradient, channels-last activations -- against torch's convolution in fp64 on the CPU."""
import pytest
import torch
import torch.nn as nn

from gpu_util import DEV, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,ci,h,co,k,s,p,ws", [(1, 1, 3, 1, 1, 1, 0, 1), (2, 33, 9, 66, 3, 2, 1, 2), (3, 32, 12, 32, 3, 1, 0, 4),
                                                (1, 65, 7, 40, 5, 1, 2, 8), (5, 4, 17, 24, 3, 3, 1, 3), (9, 64, 20, 130, 1, 1, 0, 2)])
def test_tiles_against_torch(n, ci, h, co, k, s, p, ws, dtype):
    from rtp_amd import emulate_shards
    from rtp_amd.module.conv import ColumnParallelConv2d
    gen = torch.Generator().manual_seed(co + k)
    ref = nn.Conv2d(ci, co, k, s, p)
    with torch.no_grad():
        for q in ref.parameters():
            q.copy_(torch.randn(q.shape, generator=gen).to(dtype))
    with emulate_shards(ws):
        layer = ColumnParallelConv2d(ci, co, k, s, p, device=DEV, dtype=dtype, Conv2d_layer=ref)
    x = torch.randn(n, ci, h, h, generator=gen).to(dtype)
    ref = ref.double()
    for fmt in (torch.contiguous_format, torch.channels_last):
        xd = x.to(DEV).contiguous(memory_format=fmt).requires_grad_()
        y = layer(xd)
        g = torch.randn(y.shape, generator=gen).to(dtype)
        layer.zero_grad()
        y.backward(g.to(DEV).contiguous(memory_format=fmt))
        xr = x.double().requires_grad_()
        ref.zero_grad()
        yr = ref(xr)
        yr.backward(g.double())
        assert_close(y, yr, dtype, "y")
        assert_close(xd.grad, xr.grad, dtype, "dx")
        assert_close(torch.cat([q.weight.grad for q in layer.layers]), ref.weight.grad, dtype, "dW")
        assert_close(torch.cat([q.bias.grad for q in layer.layers]), ref.bias.grad, dtype, "db")
