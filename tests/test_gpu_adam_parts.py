"""The Adam update of many buffers: chunks of every length around the parts they are dealt over, at any alignment, with the step count
from the host or from device memory, against adam_step on each buffer alone (the same arithmetic: the same bits)."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu

LENGTHS = [1, 3, 4, 1020, 1023, 1024, 1028, 4099, 16383, 16384, 16385, 40000]


@pytest.mark.parametrize("device_step", [False, True])
@pytest.mark.parametrize("offset", [0, 1, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_chunks_of_any_length(dtype, offset, device_step):
    _check(dtype, offset, device_step, sum(LENGTHS) + 100003)


@pytest.mark.parametrize("average", [0, 1500, 3000, 6000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_parts_by_the_average_chunk(dtype, average):
    """1, 2, 4 and 8 parts a chunk (16 above): what the launch is sized by changes no result."""
    _check(dtype, 1, True, average * (len(LENGTHS) + 1))


def _check(dtype, offset, device_step, total):
    from rtp_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(offset)

    def buffer(n, dt, scale=1.0):
        return (torch.randn(n + 8, generator=gen, device=DEV) * scale).to(dt)[offset:offset + n]

    step = torch.tensor([7], dtype=torch.int64, device=DEV) if device_step else 7
    sets = []
    for n in LENGTHS:
        master, grad, m = buffer(n, torch.float32), buffer(n, dtype, 0.1), buffer(n, torch.float32, 0.01)
        v = buffer(n, torch.float32, 0.01).abs()
        shadow = master.to(dtype) if dtype != torch.float32 else None
        sets.append((master, grad, shadow, m, v))
    alone = [tuple(None if t is None else t.clone() for t in s) for s in sets]
    table = ops.adam_chunk_table(sets, DEV)
    # and one chunk longer than the optimisers make them
    long = [buffer(100003, torch.float32), buffer(100003, dtype, 0.1), None, buffer(100003, torch.float32, 0.01),
            buffer(100003, torch.float32, 0.01).abs()]
    alone.append(tuple(None if t is None else t.clone() for t in long))
    row = [0 if t is None else t.data_ptr() for t in long] + [100003]
    table = torch.cat([table, torch.tensor([row], dtype=torch.int64, device=DEV)])
    ops.adam_step_multi(table, dtype, step, 1e-3, (0.9, 0.999), 1e-8, 0.01, 0.05, total)
    for got, want in zip(sets + [tuple(long)], alone):
        master, grad, shadow, m, v = want
        ops.adam_step(master, grad.contiguous(), shadow, m, v, step, 1e-3, (0.9, 0.999), 1e-8, 0.01, 0.05)
        for a, b in zip(got, want):
            assert a is None or torch.equal(a, b)


def test_more_chunks_than_one_launch_deals_over_parts():
    """2^20 chunks: sixteen workgroups each would be a launch of 2^32 threads, which is one too many."""
    from rtp_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(3)
    chunks, n = 1 << 20, 3
    total = chunks * n
    bufs = [torch.randn(total, generator=gen, device=DEV) * s for s in (1.0, 0.1, 0.01, 0.01)]
    bufs[3].abs_()
    want = [b.clone() for b in bufs]
    first = torch.arange(chunks, dtype=torch.int64, device=DEV) * (4 * n)
    master, grad, m, v = (b.data_ptr() + first for b in bufs)
    table = torch.stack([master, grad, torch.zeros_like(first), m, v, torch.full_like(first, n)], dim=1).contiguous()
    ops.adam_step_multi(table, torch.float32, 7, 1e-3, (0.9, 0.999), 1e-8, 0.01, 0.05, total)
    ops.adam_step(want[0], want[1], None, want[2], want[3], 7, 1e-3, (0.9, 0.999), 1e-8, 0.01, 0.05)
    for a, b in zip(bufs, want):
        assert torch.equal(a, b)
