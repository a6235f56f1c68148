"""The two-launch embedding backward (ids grouped by table row) against the sort and scatter-add: bit for bit at the edges of
its parts -- a row's positions around the 64 from which it is dealt over columns, the 8192-position windows of a long row,
tables smaller than the grouping pass's slices, unaligned columns -- and the gather over all shards of a token."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,table_f32", [(torch.float32, False), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("n,vocab,cols,groups,same", [(1, 9, 8, 1, 0), (200, 40, 33, 2, 63), (200, 7, 512, 4, 64),
                                                      (300, 5000, 16, 1, 65), (8193, 300, 24, 3, 8192),
                                                      (20000, 9000, 264, 2, 9000), (700, 3, 7, 1, 700)])
def test_grouped_backward_equals_sort_and_scatter(dtype, table_f32, n, vocab, cols, groups, same):
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(n + cols)
    ids = torch.randint(0, vocab, (n,), generator=gen)
    ids[torch.randperm(n, generator=gen)[:same]] = vocab // 2       # one frequent id
    g = torch.randn(n, groups * cols, generator=gen).to(dtype).to(DEV)
    tdt = torch.float32 if table_f32 else dtype
    row_begin, rows = (vocab // 4, vocab // 2) if vocab >= 8 else (0, vocab)
    start = torch.randn(groups, rows, cols, generator=gen).to(tdt).to(DEV)
    dev_ids = ids.to(DEV)
    ws = ops.embedding_sort_ids(dev_ids)
    for zero_fill, by_freq, scale, pad in ((True, False, 1.0, -1), (False, False, 1.0, int(ids[0])), (True, True, 0.25, -1),
                                           (False, True, 3.0, int(ids[-1]))):
        a, b = start.clone(), start.clone()
        kw = dict(row_begin=row_begin, padding_idx=pad, scale_by_freq=by_freq, zero_fill=zero_fill, groups=groups,
                  grad_out_sg=cols, grad_table_sg=rows * cols, grad_scale=scale)
        ops.embedding_scatter_add(g[:, :cols], n, ws, a[0], **kw)
        ops.embedding_backward(g[:, :cols], dev_ids, b[0], grouped=True, **kw)
        torch.cuda.synchronize()
        assert torch.equal(a, b), f"zero_fill={zero_fill} by_freq={by_freq} scale={scale} pad={pad}"
    if table_f32:
        return
    # the update where the row's gradient is produced
    masters = [torch.randn(groups, rows, cols, generator=torch.Generator().manual_seed(3)).to(DEV) for _ in range(2)]
    weights = [m.to(dtype) for m in masters]
    sgd = ops.FusedSgd(0.1, 0.05)
    for grouped, m, w in ((False, *[v[0] for v in (masters, weights)]), (True, *[v[1] for v in (masters, weights)])):
        out = start.clone()
        kw = dict(row_begin=row_begin, groups=groups, grad_out_sg=cols, grad_table_sg=rows * cols, sgd=sgd,
                  sgd_master=m.data_ptr(), sgd_weights=0 if dtype == torch.float32 else w.data_ptr())
        if grouped:
            ops.embedding_backward(g[:, :cols], dev_ids, out[0], grouped=True, **kw)
        else:
            ops.embedding_scatter_add(g[:, :cols], n, ws, out[0], **kw)
        torch.cuda.synchronize()
        assert torch.equal(out, start)
    assert torch.equal(masters[0], masters[1]) and torch.equal(weights[0], weights[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,cols,groups", [(1, 8, 1), (5, 24, 3), (7, 1032, 2), (6, 33, 4)])
def test_gather_over_shards(dtype, n, cols, groups):
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(cols)
    table = torch.randn(groups, 50, cols, generator=gen).to(dtype).to(DEV)
    pos = torch.randn(4, groups * cols, generator=gen).to(dtype).to(DEV)
    ids = torch.randint(0, 50, (n,), generator=gen).to(DEV)
    want = table[:, ids].permute(1, 0, 2).reshape(n, groups * cols)
    out = torch.empty_like(want)
    kw = dict(groups=groups, table_sg=50 * cols, out_sg=cols)
    ops.embedding_gather(table[0], ids, out[:, :cols], **kw)
    assert torch.equal(out, want)
    ops.embedding_gather(table[0], ids, out[:, :cols], scale=3.0, pos=pos[:, :cols], pos_sg=cols, batch=2, **kw)
    assert torch.equal(out, want * 3.0 + pos[torch.arange(n, device=DEV) // 2])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("scale", [1.0, 0.5])
@pytest.mark.parametrize("n,cols,groups", [(2300, 300, 1), (9000, 40, 3)])
def test_long_rows(dtype, scale, n, cols, groups):
    """Rows of every length around the blocks of 16 and rounds of 64 that a long row is summed in, the 32 positions from which
    a row is dealt over columns and the 512 from which its positions are listed by windows; columns that end inside a workgroup."""
    from rtp_amd import ops
    gen = torch.Generator().manual_seed(n)
    counts = [1, 3, 4, 5, 15, 16, 31, 32, 33, 47, 48, 49, 63, 64, 65, 127, 511, 512, 513]
    ids = torch.cat([torch.full((c,), r) for r, c in enumerate(counts)])
    ids = torch.cat([ids, torch.full((n - ids.numel(),), len(counts))])[torch.randperm(n, generator=gen)].to(DEV)
    rows = len(counts) + 2
    g = torch.randn(n, groups * cols, generator=gen).to(dtype).to(DEV)
    ws = ops.embedding_sort_ids(ids)
    a, b = (torch.full((groups, rows, cols), 7.0, dtype=dtype, device=DEV) for _ in range(2))
    kw = dict(row_begin=0, zero_fill=True, groups=groups, grad_out_sg=cols, grad_table_sg=rows * cols, grad_scale=scale)
    ops.embedding_scatter_add(g[:, :cols], n, ws, a[0], **kw)
    ops.embedding_backward(g[:, :cols], ids, b[0], grouped=True, **kw)
    assert torch.equal(a, b)
