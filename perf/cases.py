"""The work that is timed when this framework is made faster: calls of its public entry points as a training program
makes them, over the range of sizes, types and options in use.

listed() names the cases, draw(rng) gives more of the same ranges, prepare(case, seed) makes what a program has in hand
before the call, run(state) is one pass, work(case) what a pass cannot do without and tolerance(case) how far two correct
implementations may be apart.  Layers are called eagerly, gradients start at None as after an optimiser's zero_grad(); the
language model's step is called eagerly or replayed from a captured HIP graph, as bench.py does.

Ranges (draw):
  linear     1 - 8192 token rows, widths 64 - 8192 (a half multiples of 64, a quarter of 8, a quarter any that the shard
             count divides), column or row shards, 1 - 8 of them, bf16 or fp32, forward alone or with backward
  embedding  64 - 65536 ids over a vocabulary of 1000 - 50000, uniform or word-frequency (1 / rank) ids, width 128 - 4096
  attention  16 - 2048 queries, head dimension 32 / 64 / 128, 1 - 32 heads, causal, padded or plain self-attention, or
             keys and values of another sequence, bf16 or fp32
  moe        8 or 16 experts in 8 shards, 64 - 4096 tokens, d_model 128 - 2048, d_ff 256 - 8192, bf16 or fp32
  conv       1 - 64 channels in, 8 - 128 out, kernels 1 / 3 / 5, images 7 - 64 wide, batch 1 - 128, bf16 or fp32
  lm         the transformer language model of 1 - 10 blocks, width 128 - 2048, 8 - 128 positions, SGD or Adam, or the
             forward pass alone; eager or replayed
"""
import math

import torch

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
_DEV = "cuda:0"


def listed():
    return [
        # the smallest call: one sequence's hidden states through a small layer, as in evaluation; launches and host work
        {"name": "linear_small_forward", "kind": "linear", "style": "column", "rows": 32, "n_in": 256, "n_out": 256,
         "shards": 2, "dtype": "bf16", "backward": False},
        # BASELINE configuration 1
        {"name": "linear_column_fp32", "kind": "linear", "style": "column", "rows": 1024, "n_in": 2048, "n_out": 2048,
         "shards": 2, "dtype": "fp32", "backward": True},
        # what the wrapper makes of a head whose class count the shard count does not divide: row shards, an odd width;
        # the token count is the reference loop's (31 positions x 32 sequences)
        {"name": "linear_row_odd_bf16", "kind": "linear", "style": "row", "rows": 992, "n_in": 2048, "n_out": 1001,
         "shards": 8, "dtype": "bf16", "backward": True},
        # BASELINE configuration 2
        {"name": "embedding_fp32", "kind": "embedding", "vocab": 10240, "width": 2048, "shards": 4, "ids": 1024,
         "ids_like": "uniform", "dtype": "fp32", "backward": True},
        # a long step of running text: word frequencies, an odd sequence length
        {"name": "embedding_text_bf16", "kind": "embedding", "vocab": 10240, "width": 2048, "shards": 8, "ids": 1023 * 16,
         "ids_like": "text", "dtype": "bf16", "backward": True},
        # BASELINE configuration 3
        {"name": "attention_causal_bf16", "kind": "attention", "length": 512, "keys": 512, "batch": 8, "heads": 32,
         "head_dim": 64, "shards": 8, "mode": "causal", "dtype": "bf16", "backward": True},
        # encoder attention over long padded sequences of an odd length, the wider heads
        {"name": "attention_padded_bf16", "kind": "attention", "length": 1500, "keys": 1500, "batch": 4, "heads": 16,
         "head_dim": 128, "shards": 4, "mode": "padded", "dtype": "bf16", "backward": True},
        # a decoder's attention over the encoder's states, in the reference's default type
        {"name": "attention_cross_fp32", "kind": "attention", "length": 100, "keys": 180, "batch": 16, "heads": 8,
         "head_dim": 64, "shards": 4, "mode": "cross", "dtype": "fp32", "backward": True},
        # BASELINE configuration 5
        {"name": "moe_bf16", "kind": "moe", "tokens": 4096, "d_model": 2048, "d_ff": 8192, "experts": 8, "shards": 8,
         "dtype": "bf16", "backward": True},
        # the second convolution of the MNIST network of the reference's demo
        {"name": "conv_mnist_fp32", "kind": "conv", "batch": 64, "c_in": 32, "c_out": 64, "size": 26, "kernel": 3,
         "stride": 1, "padding": 0, "shards": 4, "dtype": "fp32", "backward": True},
        # BASELINE configuration 4, the headline: one training step replayed from a captured graph
        {"name": "lm_step_replayed", "kind": "lm", "vocab": 10240, "width": 2048, "hidden": 2048, "heads": 32,
         "layers": 10, "length": 32, "batch": 32, "shards": 8, "dtype": "bf16", "step": "sgd", "graph": True},
        # the reference's own loop on the same model: 31 x 32 tokens, clip + Adam, called eagerly
        {"name": "lm_step_eager_adam", "kind": "lm", "vocab": 10240, "width": 2048, "hidden": 2048, "heads": 32,
         "layers": 10, "length": 31, "batch": 32, "shards": 8, "dtype": "bf16", "step": "adam", "graph": False},
    ]


# ---- drawn cases ----


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 1e-9))))


def _width(rng, lo, hi, unit):
    """A width in lo .. hi that `unit` divides: half of them multiples of 64, a quarter of 8, a quarter of `unit` alone."""
    step = math.lcm(unit, rng.choice((64, 64, 8, 1)))
    return max(step, _log(rng, lo, hi) // step * step)


def _draw_once(rng):
    kind = rng.choice(("linear", "linear", "linear", "embedding", "embedding", "attention", "attention", "attention",
                       "moe", "conv", "lm", "lm"))
    ws = rng.choice((1, 2, 4, 8))
    dtype = rng.choice(("bf16", "bf16", "fp32"))
    backward = rng.random() < 0.75
    if kind == "linear":
        column = rng.random() < 0.6
        return {"kind": kind, "style": "column" if column else "row", "rows": _log(rng, 1, 8192),
                "n_in": _width(rng, 64, 8192, 1 if column else ws), "n_out": _width(rng, 64, 8192, ws if column else 1),
                "shards": ws, "dtype": dtype, "backward": backward}
    if kind == "embedding":
        return {"kind": kind, "vocab": _log(rng, 1000, 50000), "width": _width(rng, 128, 4096, 8 * ws), "shards": ws,
                "ids": _log(rng, 64, 65536), "ids_like": rng.choice(("uniform", "text")), "dtype": dtype,
                "backward": backward}
    if kind == "attention":
        mode = rng.choice(("causal", "causal", "padded", "plain", "cross"))
        length = _log(rng, 16, 2048)
        return {"kind": kind, "length": length, "keys": _log(rng, 16, 2048) if mode == "cross" else length,
                "batch": _log(rng, 1, 32), "heads": ws * rng.choice((1, 2, 4)), "head_dim": rng.choice((32, 64, 64, 128)),
                "shards": ws, "mode": mode, "dtype": dtype, "backward": backward}
    if kind == "moe":
        experts = rng.choice((8, 16))
        return {"kind": kind, "tokens": max(64, _log(rng, 64, 4096) // experts * experts),
                "d_model": _width(rng, 128, 2048, 64), "d_ff": _width(rng, 256, 8192, 64), "experts": experts,
                "shards": 8, "dtype": dtype, "backward": True}
    if kind == "conv":
        kernel = rng.choice((1, 3, 3, 5))
        return {"kind": kind, "batch": _log(rng, 1, 128), "c_in": _log(rng, 1, 64), "c_out": ws * _log(rng, 8, 128 // ws),
                "size": rng.randint(7, 64), "kernel": kernel, "stride": rng.choice((1, 1, 2)),
                "padding": rng.choice((0, kernel // 2)), "shards": ws, "dtype": dtype, "backward": backward}
    head_dim = rng.choice((32, 64, 64, 128))
    heads = ws * max(1, _log(rng, 128, 2048) // (head_dim * ws))
    return {"kind": kind, "vocab": ws * _log(rng, 64, 32768 // ws), "width": heads * head_dim,
            "hidden": ws * _log(rng, 16, 4096 // ws), "heads": heads, "layers": rng.randint(1, 10),
            "length": _log(rng, 8, 128), "batch": _log(rng, 1, 64), "shards": ws, "dtype": dtype,
            "step": rng.choice(("sgd", "adam", "forward")), "graph": rng.random() < 0.5}


def _cost(case):
    """Operations, an fp32 one counted as 16 of bf16 (the ratio of the matrix peaks), and a byte as 300."""
    w = work(case)
    return w["flops"] * (16 if case["dtype"] == "fp32" else 1) + 300 * w["bytes"]


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw_once(rng)
        if c["kind"] == "attention" and c["batch"] * c["heads"] * c["length"] * c["keys"] > 1 << 27:
            continue  # the fp32 form keeps the probabilities
        if c["kind"] == "conv" and work(c)["flops"] > 3e10:
            continue
        if c["kind"] == "lm" and c["length"] * c["batch"] > 2048:
            continue
        if _cost(c) <= most:
            return c


# ---- states ----


def _fill(gen, shape, dtype, lo=None, hi=None):
    t = torch.empty(shape, dtype=torch.float32, device=_DEV)
    t = t.normal_(generator=gen) if lo is None else t.uniform_(lo, hi, generator=gen)
    return t.to(dtype)


def _token_ids(gen, count, vocab, like):
    """Uniform ids (the benchmark's), or ids by word frequency: the chance of the word of rank r is ~ 1 / r."""
    u = torch.rand(count, generator=gen, device=_DEV, dtype=torch.float64)
    ids = torch.floor(u * vocab) if like == "uniform" else torch.floor(torch.exp(u * math.log(vocab + 1))) - 1
    return ids.to(torch.int64).clamp_(0, vocab - 1)


def _weights(layer, gen):
    """Every parameter ~ U(-0.1, 0.1), as the reference's initrange and this repository's configurations have it."""
    with torch.no_grad():
        for p in layer.parameters():
            p.uniform_(-0.1, 0.1, generator=gen)


def prepare(case, seed):
    torch.manual_seed(seed)
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    return _PREPARE[case["kind"]](case, gen, _DTYPES[case["dtype"]])


def _layer_state(case, layer, gen, inputs, kwargs, out_shape, dtype):
    _weights(layer, gen)
    backward = case["backward"]
    state = {"layer": layer, "inputs": inputs, "kwargs": kwargs, "backward": backward,
             "leaves": [t for t in inputs if backward and t.is_floating_point()],
             "params": list(layer.parameters()), "dy": _fill(gen, out_shape, dtype) if backward else None}
    for t in state["leaves"]:
        t.requires_grad_()
    return state


def _prepare_linear(case, gen, dtype):
    from rtp_amd import emulate_shards
    from rtp_amd.module.linear import ColumnParallelLinear, RowParallelLinear
    cls = ColumnParallelLinear if case["style"] == "column" else RowParallelLinear
    with emulate_shards(case["shards"]):
        layer = cls(case["n_in"], case["n_out"], device=_DEV, dtype=dtype)
    x = _fill(gen, (case["rows"], case["n_in"]), dtype)
    return _layer_state(case, layer, gen, [x], {}, (case["rows"], case["n_out"]), dtype)


def _prepare_embedding(case, gen, dtype):
    from rtp_amd.module.embedding import ParallelEmbedding
    layer = ParallelEmbedding(case["vocab"], case["width"], case["shards"], 0, device=_DEV, dtype=dtype)
    ids = _token_ids(gen, case["ids"], case["vocab"], case["ids_like"])
    return _layer_state(case, layer, gen, [ids], {}, (case["ids"], case["width"]), dtype)


def _prepare_attention(case, gen, dtype):
    from rtp_amd.module.attention import ParallelMultiheadAttention
    width = case["heads"] * case["head_dim"]
    layer = ParallelMultiheadAttention(width, case["heads"], case["shards"], 0, device=_DEV, dtype=dtype)
    x = _fill(gen, (case["length"], case["batch"], width), dtype)
    kwargs = {"need_weights": False}
    inputs = [x]
    if case["mode"] == "causal":
        kwargs["is_causal"] = True
    elif case["mode"] == "padded":  # sequences of unequal length: between a half and all of the positions are real
        real = torch.randint(case["length"] // 2 + 1, case["length"] + 1, (case["batch"], 1), generator=gen, device=_DEV)
        kwargs["key_padding_mask"] = torch.arange(case["length"], device=_DEV)[None, :] >= real
    elif case["mode"] == "cross":
        inputs.append(_fill(gen, (case["keys"], case["batch"], width), dtype))
    return _layer_state(case, layer, gen, inputs, kwargs, x.shape, dtype)


def _prepare_moe(case, gen, dtype):
    from rtp_amd import emulate_shards
    from rtp_amd.models.transformer_lm_rtp import FeedForwardLayer_expert
    from rtp_amd.module.moe import WeightMOELayer
    from rtp_amd.module.top2gate import WeightTop2Gate
    m, local = case["d_model"], case["experts"] // case["shards"]
    with emulate_shards(case["shards"]):
        gate = WeightTop2Gate(m, case["experts"], device=_DEV, dtype=dtype)
        experts = torch.nn.ModuleList([FeedForwardLayer_expert(m, case["d_ff"], torch.nn.ReLU(), 0.0, device=_DEV,
                                                               dtype=dtype) for _ in range(local)])
        layer = WeightMOELayer(gate, experts, device=_DEV, dtype=dtype)
    x = _fill(gen, (8, case["tokens"] // 8, m), dtype)
    u = torch.rand(case["tokens"], case["experts"], generator=gen, device=_DEV).clamp_(1e-7, 1 - 1e-7)
    noise = -torch.log(-torch.log(u))  # the routing noise, handed over so that a pass can be repeated
    return _layer_state(case, layer, gen, [x], {"noise": noise}, x.shape, dtype)


def _prepare_conv(case, gen, dtype):
    from rtp_amd import emulate_shards
    from rtp_amd.module.conv import ColumnParallelConv2d
    with emulate_shards(case["shards"]):
        layer = ColumnParallelConv2d(case["c_in"], case["c_out"], case["kernel"], case["stride"], case["padding"],
                                     device=_DEV, dtype=dtype)
    x = _fill(gen, (case["batch"], case["c_in"], case["size"], case["size"]), dtype)
    out = _conv_out(case)
    return _layer_state(case, layer, gen, [x], {}, (case["batch"], case["c_out"], out, out), dtype)


def _prepare_lm(case, gen, dtype):
    from rtp_amd import ring
    from rtp_amd.models.transformer_lm_rtp import TransformerLM
    from rtp_amd.optim import RotatedAdam, RotatedSGD
    lm = TransformerLM(case["vocab"], case["width"], case["heads"], case["hidden"], 0.0, 0.1, case["layers"],
                       case["shards"], 0, device=_DEV, dtype=dtype)
    opt = None
    if case["step"] == "sgd":  # bench.py's: the update in the epilogue of the weight-gradient products
        opt = RotatedSGD(lm, lr=1e-3, clip_value=0.05, fused_backward=True)
    elif case["step"] == "adam":  # the reference harness's clip, and its optimiser
        opt = RotatedAdam(lm, lr=1e-4, clip_value=0.05)
    tokens = case["length"] * case["batch"]
    batch = _token_ids(gen, 2 * tokens, case["vocab"], "uniform").view(2, case["length"], case["batch"])
    state = {"lm": lm, "opt": opt, "batch": batch, "vocab": case["vocab"], "graph": None, "mirror": []}
    if opt is not None:
        masters = [st.home if m is None else m for st, m in zip(opt.stores, opt.masters)]
        state["mirror"] = masters + [opt.flat if opt.flat_master is None else opt.flat_master]
    if case["graph"]:
        # one step recorded as bench.py records it: eager steps on a side stream first (on a batch of their own), the
        # weight gradients of the backward pass on a second stream, then the capture
        ring.set_wgrad_overlap(opt is not None)
        state["static"] = _token_ids(gen, 2 * tokens, case["vocab"], "uniform").view_as(batch)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                _lm_pass(state, state["static"])
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        ring.fence()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["out"] = _lm_pass(state, state["static"])
        ring.fence()
        ring.set_wgrad_overlap(False)
        state["graph"] = graph
    return state


_PREPARE = {"linear": _prepare_linear, "embedding": _prepare_embedding, "attention": _prepare_attention,
            "moe": _prepare_moe, "conv": _prepare_conv, "lm": _prepare_lm}


# ---- one pass ----


def _lm_pass(state, batch):
    from rtp_amd.module.loss import cross_entropy
    lm, opt = state["lm"], state["opt"]
    if opt is None:
        with torch.no_grad():
            return lm(batch[0])
    opt.zero_grad()
    loss = cross_entropy(lm(batch[0]).view(-1, state["vocab"]), batch[1].view(-1))
    loss.backward()
    opt.step()
    return loss.detach()


def run(state):
    if "lm" in state:
        if state["graph"] is None:
            out = _lm_pass(state, state["batch"])
        else:
            state["static"].copy_(state["batch"])
            state["graph"].replay()
            out = state["out"]
        return [out] + state["mirror"]
    layer, inputs = state["layer"], state["inputs"]
    if len(inputs) == 2:
        args = [inputs[0], inputs[1], inputs[1]]  # the encoder's states are keys and values
    else:
        args = inputs * (3 if "need_weights" in state["kwargs"] else 1)
    if not state["backward"]:
        with torch.no_grad():
            out = layer(*args, **state["kwargs"])
        return out[0] if isinstance(out, tuple) else out
    layer.zero_grad()
    for t in state["leaves"]:
        t.grad = None
    out = layer(*args, **state["kwargs"])
    if isinstance(out, tuple):
        out = out[0]
    out.backward(state["dy"])
    result = [out.detach()] + [t.grad for t in state["leaves"]] + [p.grad for p in state["params"]]
    l_aux = getattr(layer, "l_aux", None)
    return result if l_aux is None else result + [l_aux.detach()]


# ---- what a pass cannot do without ----


def _conv_out(case):
    return (case["size"] + 2 * case["padding"] - case["kernel"]) // case["stride"] + 1


def work(case):
    kind, es = case["kind"], 2 if case["dtype"] == "bf16" else 4
    if kind == "lm":
        tokens, width = case["length"] * case["batch"], case["width"]
        block = 4 * width * width + 2 * width * case["hidden"]
        matrices = case["layers"] * block + width * case["vocab"]
        core = 4.0 * case["layers"] * case["batch"] * case["length"] ** 2 * width * 0.5  # causal
        flops = 2.0 * tokens * matrices + core
        params = matrices + width * case["vocab"]
        logits = es * tokens * case["vocab"]
        if case["step"] == "forward":
            return {"flops": flops, "bytes": es * matrices + es * tokens * width + logits}
        # SGD reads and writes the parameters (and, in bf16, their fp32 masters) of every matrix, and the table rows that
        # the step names; Adam everything, with two moments
        shadow = 0 if es == 4 else 4
        if case["step"] == "sgd":
            return {"flops": 3 * flops, "bytes": (8 + shadow) * (matrices + min(tokens, case["vocab"]) * width)}
        return {"flops": 3 * flops, "bytes": (24 + shadow) * params}
    passes = 3 if case["backward"] else 1
    if kind == "linear":
        r, k, n = case["rows"], case["n_in"], case["n_out"]
        forward = r * k + n * k + n + r * n
        return {"flops": 2.0 * passes * r * k * n,
                "bytes": es * (2 * forward if case["backward"] else forward)}
    if kind == "embedding":
        t, d, v = case["ids"], case["width"], case["vocab"]
        forward = es * 2 * t * d + 8 * t
        return {"flops": float(t * d), "bytes": forward + (es * (t * d + v * d) if case["backward"] else 0)}
    if kind == "attention":
        l, s, n, e = case["length"], case["keys"], case["batch"], case["heads"] * case["head_dim"]
        inputs = l * n * e + (s * n * e if case["mode"] == "cross" else 0)
        visible = 0.5 if case["mode"] == "causal" else 1.0
        flops = 4.0 * n * e * e * (l + s) + 4.0 * n * l * s * e * visible
        once = inputs + l * n * e + 4 * e * e + 4 * e
        return {"flops": passes * flops, "bytes": es * (2 * once if case["backward"] else once)}
    if kind == "moe":
        t, m, f, ex = case["tokens"], case["d_model"], case["d_ff"], case["experts"]
        return {"flops": 3 * 2.0 * 2 * t * 2 * m * f, "bytes": es * 2 * (2 * t * m + ex * (2 * m * f + m + f) + ex * m)}
    out, k2 = _conv_out(case), case["kernel"] ** 2
    forward = case["batch"] * (case["c_in"] * case["size"] ** 2 + case["c_out"] * out * out) + \
        case["c_out"] * (case["c_in"] * k2 + 1)
    return {"flops": 2.0 * passes * case["batch"] * out * out * case["c_out"] * case["c_in"] * k2,
            "bytes": es * (2 * forward if case["backward"] else forward)}


def tolerance(case):
    """bf16 results are rounded to 8 bits at every layer's border, fp32 sums differ by their order.  The gather is a copy
    and the sums of an embedding's gradient have a fixed order: exact.  A training step carries its rounding through
    every block and on into the signs that Adam's first updates consist of."""
    if case["kind"] == "embedding":
        return "exact"
    if case["kind"] == "lm":
        bf16 = case["dtype"] == "bf16"
        if case["step"] == "forward":
            return {"rel": 2e-2, "max": 0.3} if bf16 else {"rel": 1e-4, "max": 5e-3}
        if case["step"] == "adam":
            return {"rel": 1e-2, "max": 0.1} if bf16 else {"rel": 1e-3, "max": 0.1}
        return {"rel": 2e-3, "max": 2e-2} if bf16 else {"rel": 1e-4, "max": 1e-2}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 2e-5, "max": 1e-3} if case["kind"] in ("attention", "moe") else {"rel": 1e-5, "max": 5e-4}
