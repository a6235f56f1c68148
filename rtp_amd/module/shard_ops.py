"""Grouped launches over a run of consecutive shards staged as `flat` = [count, numel].

A weight matrix of the layer is described by (offset inside a flat shard, rows, cols); shard g of the run
is found `numel` elements after shard g-1, which is the group / K-segment stride handed to rtp_gemm.
Column-style matrices (output features sharded) use one group per shard; row-style matrices (input
features sharded) contract over the shards as K segments, so their cross-shard sum stays in the MFMA
accumulators.
"""
from __future__ import annotations

from typing import Optional

import torch

from .. import _lib, ops, ring


_ROWSUM_DONE, _SGD_DONE = 1, 2  # of native().gemm and its relatives


def _rows(t: torch.Tensor):
    m, n, ld = ops._mat(t, "operand")
    return m, n, ld


def col_fwd(x2, flat, w_off, n_s, k, bias_off, out, col0, *, relu=False):
    """out[:, col0 + g*n_s : col0 + (g+1)*n_s] = x2 @ W_g^T (+ b_g), g over the run: the run is a rotated
    column-parallel layer of its own (rtp_rotated_linear_fwd) whose outputs start at column col0."""
    ops.native().linear_fwd(x2, flat, w_off, bias_off, n_s, k, out, col0, relu)


def col_dgrad(dy2, flat, w_off, n_s, k, out, col0, c_in: Optional[torch.Tensor] = None, gate=None):
    """out[M, k] = (c_in +) sum_g dy2[:, col0 + g*n_s : ...] @ W_g   (contraction segmented over shards)."""
    ops.native().linear_bwd(dy2, col0, None, flat, w_off, None, n_s, k, out, c_in, gate, None, False, None, None, 0.0, 0.0,
                            False)


def _fused(store, accumulate, first, cnt, w_off, length):
    """Keyword arguments that make a weight-gradient product of `store` apply the optimiser's update itself (when
    an optimiser has asked for that, RotatedSGD(fused_backward=True)), and the note of what it covers."""
    f = getattr(store, "fused_sgd", None) if store is not None else None
    if f is None:
        return {}
    if accumulate:
        raise RuntimeError("RotatedSGD(fused_backward=True): a rotated layer produced gradients twice before step(); "
                           "use fused_backward=False for gradient accumulation or shared layers")
    return f.bind(store, first, cnt, w_off, length)


def _fused_done(store, kw):
    """After the launch: if the library could not fuse the update for these operands, take the note back (the
    optimiser then updates that range itself)."""
    if kw:
        store.fused_sgd.confirm()


def col_wgrad(dy2, x2, grads, first, w_off, n_s, k, col0, cnt, accumulate, b_off: Optional[int] = None, store=None):
    """grads[first+g, w_off : w_off + n_s*k] (+)= dy2[:, col0 + g*n_s : ...]^T @ x2, g < cnt; with `b_off` also the
    bias gradients grads[first+g, b_off : b_off + n_s] (+)= column sums of the same block of dy2.  `store`: the
    layer's ShardStore, for an optimiser that applies its update inside this launch."""
    es = grads.element_size()
    if n_s == 1 and cnt > 1:
        numel = grads.shape[1]
        m, _, lda = _rows(dy2)
        _, _, ldb = _rows(x2)
        c = grads.data_ptr() + (first * numel + w_off) * es
        # one output row per shard (a gate with one expert per shard): the run is a single product whose
        # output rows are the shards' gradient rows, `numel` apart -- vector loads instead of 1-row groups
        ops.gemm_raw(grads.dtype, a=dy2.data_ptr() + col0 * es, b=x2.data_ptr(), c_out=c, m=cnt, n=k, k=m, lda=lda,
                     ldb=ldb, ldc=numel, a_kcontig=False, b_kcontig=False,
                     c_in=c if accumulate else None, ld_cin=numel, stream_out=True)
        if b_off is not None:
            col_bgrad(dy2, grads, first, b_off, n_s, col0, cnt, accumulate)
        return
    # one launch for the run (rtp_rotated_linear_bwd): the weight gradients, the bias gradients as the row sums of the
    # product's first operand dy^T, and the optimiser's update where one asked for it
    kw = _fused(store, accumulate, first, cnt, w_off, n_s * k)
    # the weight-gradient half reads no weights: the gradient rows give the layout
    run = grads if cnt == grads.shape[0] else grads[first:first + cnt]
    if kw:  # bound to the weight's own address; the entry point takes the run's base and adds w_off itself
        sgd = kw["sgd"]
        done = ops.native().linear_bwd(dy2, col0, x2, run, w_off, b_off, n_s, k, None, None, None, run, accumulate,
                                       kw["sgd_master"] - w_off * 4,
                                       kw["sgd_weights"] - w_off * es if kw["sgd_weights"] else None, sgd.lr, sgd.clip,
                                       not sgd.keep_grads)
    else:
        done = ops.native().linear_bwd(dy2, col0, x2, run, w_off, b_off, n_s, k, None, None, None, run, accumulate, None,
                                       None, 0.0, 0.0, False)
    if kw:
        if not done & _lib.ROTATED_SGD_DONE:
            kw["sgd"].missed = True
        _fused_done(store, kw)
    if b_off is not None and not done & _lib.ROTATED_BIAS_DONE:
        col_bgrad(dy2, grads, first, b_off, n_s, col0, cnt, accumulate)


def col_bgrad(dy2, grads, first, b_off, n_s, col0, cnt, accumulate):
    """grads[first+g, b_off : b_off+n_s] (+)= column sums of dy2[:, col0 + g*n_s : ...]."""
    numel = grads.shape[1]
    block = dy2[:, col0:col0 + cnt * n_s]
    ops.colsum(block, grads[first, b_off:b_off + n_s], accumulate=accumulate, seg=n_s, seg_stride=numel)


def row_fwd(x2, flat, w_off, n, k_s, bias_off, out, col0, c_in: Optional[torch.Tensor] = None):
    """out[M, n] = (c_in +) sum_g x2[:, col0 + g*k_s : ...] @ W_g^T + sum_g b_g."""
    ops.native().row_fwd(x2, flat, w_off, bias_off, n, k_s, out, col0, c_in)


def row_dgrad(dy2, flat, w_off, n, k_s, out, col0):
    """out[:, col0 + g*k_s : ...] = dy2 @ W_g, g over the run."""
    ops.native().row_dgrad(dy2, flat, w_off, n, k_s, out, col0)


def row_wgrad(dy2, x2, grads, first, w_off, n, k_s, col0, cnt, accumulate, b_off: Optional[int] = None, store=None):
    """grads[first+g, w_off : w_off + n*k_s] (+)= dy2^T @ x2[:, col0 + g*k_s : ...]; with `b_off` also the bias
    gradients grads[first+g, b_off : b_off + n] (+)= column sums of dy2 (every shard of a row-style layer stores
    bias/ws and receives the full sum, tests/test_linear.py:181-186)."""
    kw = _fused(store, accumulate, first, cnt, w_off, n * k_s)
    if kw:
        sgd = kw["sgd"]
        done = ops.native().row_wgrad(dy2, x2, grads, first, w_off, b_off, n, k_s, col0, cnt, accumulate, kw["sgd_master"],
                                      kw["sgd_weights"] or None, sgd.lr, sgd.clip, not sgd.keep_grads)
        if not done & _lib.ROTATED_SGD_DONE:
            sgd.missed = True
        _fused_done(store, kw)
    else:
        done = ops.native().row_wgrad(dy2, x2, grads, first, w_off, b_off, n, k_s, col0, cnt, accumulate, None, None, 0.0, 0.0,
                                      False)
    if b_off is not None and not done & _lib.ROTATED_BIAS_DONE:
        row_bgrad(dy2, grads, first, b_off, n, cnt, accumulate)


def attention_wgrad(dout2, o, dqkv, x2, store, first, cnt, accumulate, w_o_off, b_o_off, E, e_s, b_in_off):
    """row_wgrad of an attention layer's out-projection and col_wgrad of its in-projection (rows q, k, v at offset 0 of a shard),
    in one launch where that is faster."""
    grads, parts = store.grads, ((w_o_off, E * e_s), (0, 3 * e_s * E))
    kws = [_fused(store, accumulate, first, cnt, *p) for p in parts]
    # Beside the input gradients on another stream the CUs that a round leaves idle are in use, and two updates at once hold that stream up:
    # replayed LM step 3690 us apart, 3716 together (without updates 4882 / 4870; on one stream 3863 / 3729).
    apart = bool(kws[0]) and ring.wgrad_overlap()
    if kws[0]:
        sgd = kws[0]["sgd"]
        weights = tuple(kw["sgd_weights"] for kw in kws)
        update = (tuple(kw["sgd_master"] for kw in kws), weights if weights[0] else None, sgd.lr, sgd.clip, not sgd.keep_grads)
    else:
        update = (None, None, 0.0, 0.0, False)
    done = ops.native().attention_wgrad(dout2, o, dqkv, x2, grads, first, cnt, accumulate, w_o_off, b_o_off, E, e_s, b_in_off, *update, apart)
    for i, p in enumerate(parts):
        if kws[0]:
            kw = _fused(store, accumulate, first, cnt, *p)
            kw["sgd"].missed = not done >> 2 * i & _SGD_DONE
            _fused_done(store, kw)
    if b_o_off is not None and not done & _ROWSUM_DONE:
        row_bgrad(dout2, grads, first, b_o_off, E, cnt, accumulate)
    if b_in_off is not None and not done >> 2 & _ROWSUM_DONE:
        col_bgrad(dqkv, grads, first, b_in_off, 3 * e_s, first * 3 * e_s, cnt, accumulate)


def row_bgrad(dy2, grads, first, b_off, n, cnt, accumulate):
    """grads[first+g, b_off : b_off + n] (+)= column sums of dy2 for every shard g of the run."""
    tmp = torch.empty(n, dtype=grads.dtype, device=grads.device)
    ops.colsum(dy2, tmp)
    dst = grads[first:first + cnt, b_off:b_off + n]
    if accumulate:
        dst.add_(tmp)
    else:
        dst.copy_(tmp.expand(cnt, n))
