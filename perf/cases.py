"""The workloads the speed of this package is measured on, each through its public functions.

A case is a dict of plain values.  Its "path" is one of
  decode   one token (or a few) through the convolutions of a stack of layers, each with its own
           weights and cache: `causal_conv1d_update`, once per layer;
  prefill  a forward without gradients: `causal_conv1d_fn`;
  handoff  a packed prefill and the decode caches of its sequences: `causal_conv1d_fwd_varlen_states`;
  train    a forward and its backward through autograd: `causal_conv1d_fn`, `torch.autograd.grad`.
Layouts of x (batch, dim, seqlen): "last" has the channels contiguous, "first" the positions,
"slice" is "last" as a window of columns of a wider projection buffer, whose rows start anywhere on
a 16-byte grid.  Every case has a bias and SiLU, as every model that uses this operator does.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "causal-conv1d_amd"))

from causal_conv1d import causal_conv1d_fn, causal_conv1d_fwd_varlen_states, causal_conv1d_update  # noqa: E402

_TYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
# Four times the relative error (2-norm) seen against the same path in 64 bits: 1.7e-3 for bf16 results and
# 2.1e-4 for fp16, their rounding; for fp32 8e-8, and 8e-7 for a sum over 32768 positions whose
# terms are added one after the other in pieces of 2048 (this package's own order: 2e-7).
_REL = {"fp32": 3e-6, "fp16": 8e-4, "bf16": 7e-3}


def _case(name, path, **values):
    return dict({"name": name, "path": path}, **values)


def listed():
    return [
        # One request generating text: a single token per layer, all launch and latency.
        _case("decode_one_request", "decode", layers=32, batch=1, dim=5376, tokens=1, width=4, state_len=4, cache="rows",
              ring=False, slots=0, dtype="bf16", weights="bf16"),
        # A decode step of a Mamba-2 2.7B-shaped model at batch 256, its cache shifted in place.
        _case("decode_batch", "decode", layers=32, batch=256, dim=5376, tokens=1, width=4, state_len=3, cache="rows",
              ring=False, slots=0, dtype="bf16", weights="fp32"),
        # A server with continuous batching: ring-buffer caches of 512 slots, a quarter of the batch padding.
        _case("decode_ring_slots", "decode", layers=32, batch=128, dim=5376, tokens=1, width=4, state_len=8, cache="rows",
              ring=True, slots=512, dtype="bf16", weights="bf16"),
        # The cache layout of Mamba blocks: (batch, dim, width), the positions of a channel adjacent.
        _case("decode_channel_cache", "decode", layers=32, batch=64, dim=5120, tokens=1, width=4, state_len=4, cache="channels",
              ring=False, slots=0, dtype="bf16", weights="bf16"),
        # One chunk of a chunked prefill: states in, states out.
        _case("prefill_chunk", "prefill", batch=1, dim=5376, seqlen=512, width=4, layout="last", seq_idx=False, states=True,
              dtype="bf16", weights="bf16"),
        # Mamba-2 2.7B-shaped prefill, 1-4 sub-sequences packed into every row.
        _case("prefill_packed", "prefill", batch=8, dim=5376, seqlen=2048, width=4, layout="last", seq_idx=True, states=False,
              dtype="bf16", weights="fp32"),
        # The forward at full precision in the positions-contiguous layout.
        _case("prefill_fp32", "prefill", batch=4, dim=2048, seqlen=4096, width=3, layout="first", seq_idx=False, states=False,
              dtype="fp32", weights="fp32"),
        # Prompts of several requests packed into one row, and the caches their decode starts from.
        _case("handoff_packed", "handoff", tokens=4096, sequences=12, dim=5376, width=4, state_len=3, dtype="bf16", weights="bf16"),
        # A small model or a unit test's training step: host work and launches.
        _case("train_small", "train", batch=2, dim=64, seqlen=512, width=4, layout="first", seq_idx=False, states=False,
              dtype="fp32", weights="fp32"),
        # Mamba-2 training: x is a window of the input projection's output, sequences packed.
        _case("train_packed_slice", "train", batch=4, dim=5376, seqlen=2048, width=4, layout="slice", seq_idx=True, states=False,
              dtype="bf16", weights="fp32"),
        # Training rows of a length that is no multiple of anything.
        _case("train_ragged", "train", batch=16, dim=4096, seqlen=1001, width=4, layout="first", seq_idx=False, states=False,
              dtype="bf16", weights="fp32"),
        # Training on long rows, with states carried in and out and their gradients.
        _case("train_long", "train", batch=4, dim=4096, seqlen=8192, width=4, layout="first", seq_idx=False, states=True,
              dtype="fp16", weights="fp32"),
    ]


_MAX_BYTES = 4 * 4096 * 8192 * 2      # of x in the largest listed case


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    path = rng.choice(["decode", "decode", "prefill", "handoff", "train", "train"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    eb = 4 if dtype == "fp32" else 2
    case = {"path": path, "dtype": dtype, "weights": rng.choice([dtype, "fp32"]), "width": rng.choice([4, 4, 4, 3, 2])}
    dim = 8 * _log_int(rng, 8, 1024) if rng.random() < 0.5 else 64 * _log_int(rng, 8, 128)
    if path == "decode":
        cache = rng.choice(["rows", "rows", "channels"])
        ring = cache == "rows" and rng.random() < 0.3
        batch = min(_log_int(rng, 1, 512), max(1, 256 * 5376 * 2 // (dim * eb)))
        tokens = 1 if cache == "channels" or rng.random() < 0.8 else rng.randint(2, 6)
        state_len = rng.choice([case["width"] - 1, case["width"], case["width"] - 1 + tokens]) if not ring else rng.choice([8, 16])
        if cache == "channels":
            state_len = case["width"]
        case.update(layers=32, batch=batch, dim=dim, tokens=tokens, state_len=max(state_len, case["width"] - 1), cache=cache,
                    ring=ring, slots=rng.choice([0, 0, 2 * batch]))
        return case
    if path == "handoff":
        tokens = min(_log_int(rng, 16, 16384), _MAX_BYTES // (dim * eb))
        case.update(tokens=tokens, sequences=_log_int(rng, 1, min(64, tokens)), dim=dim, state_len=rng.choice([3, 4]))
        return case
    seqlen = _log_int(rng, 16, 8192)
    if rng.random() < 0.5:
        seqlen = max(16, seqlen // 64 * 64)
    batch = min(_log_int(rng, 1, 32), max(1, _MAX_BYTES // (dim * seqlen * eb)))
    seqlen = min(seqlen, _MAX_BYTES // (batch * dim * eb))
    layout = rng.choice(["last", "slice", "first"])
    seq_idx = layout != "first" and rng.random() < 0.5
    case.update(batch=batch, dim=dim, seqlen=seqlen, layout=layout, seq_idx=seq_idx, states=not seq_idx and rng.random() < 0.4)
    return case


class _Maker:
    """Seeded tensors on the GPU."""

    def __init__(self, case, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev).manual_seed(seed)
        self.dtype, self.wtype = _TYPES[case["dtype"]], _TYPES[case["weights"]]

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=self.dev, dtype=self.dtype)

    def taps(self, *shape):
        return (torch.rand(*shape, generator=self.g, device=self.dev) - 0.5).to(self.wtype)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=self.dev, dtype=torch.int32)

    def x(self, batch, dim, seqlen, layout):
        if layout == "first":
            return self.normal(batch, dim, seqlen)
        if layout == "last":
            return self.normal(batch, seqlen, dim).transpose(1, 2)
        # gate | x | a few per-head values, as an input projection lays its output out
        gate, heads = dim // 16 * 16, max(8, dim // 64 // 8 * 8)
        return self.normal(batch, seqlen, gate + dim + heads)[..., gate:gate + dim].transpose(1, 2)

    def packed_ids(self, batch, seqlen):
        cuts = torch.rand(batch, 3, generator=self.g, device=self.dev) * seqlen
        cuts = torch.where(torch.rand(batch, 3, generator=self.g, device=self.dev) < 0.5, cuts, float("inf"))
        pos = torch.arange(seqlen, device=self.dev)
        return (pos.view(1, 1, -1) >= cuts.unsqueeze(-1)).sum(1).to(torch.int32)


def prepare(case, seed):
    m = _Maker(case, seed)
    dim, width = case["dim"], case["width"]
    if case["path"] == "decode":
        layers, batch, tokens, state_len = case["layers"], case["batch"], case["tokens"], case["state_len"]
        rows = case["slots"] or batch
        if case["cache"] == "rows":
            caches = m.normal(layers, rows, state_len, dim).transpose(2, 3)
        else:
            caches = m.normal(layers, rows, dim, state_len)
        if tokens == 1:
            xs = list(m.normal(layers, batch, dim).unbind(0))
        else:
            xs = list(m.normal(layers, batch, tokens, dim).transpose(2, 3).unbind(0))
        indices = lengths = None
        if case["slots"]:
            order = torch.argsort(torch.rand(rows, generator=m.g, device=m.dev))[:batch].to(torch.int32)
            padding = torch.rand(batch, generator=m.g, device=m.dev) < 0.25
            indices = torch.where(padding, torch.full_like(order, -1), order)
        if case["ring"]:
            lengths = m.ints(0, 1000, batch)
        return {"path": "decode", "xs": xs, "all_caches": caches, "caches": list(caches.unbind(0)),
                "weights": list(m.taps(layers, dim, width).unbind(0)), "biases": list(m.taps(layers, dim).unbind(0)),
                "lengths": lengths, "indices": indices}
    weight, bias = m.taps(dim, width), m.taps(dim)
    if case["path"] == "handoff":
        tokens, sequences = case["tokens"], case["sequences"]
        inner = torch.randperm(tokens - 1, generator=m.g, device=m.dev)[:sequences - 1].sort().values + 1
        ends = torch.tensor([tokens], device=m.dev)
        cu = torch.cat([torch.zeros_like(ends), inner, ends]).to(torch.int32)
        ids = torch.bucketize(torch.arange(tokens, device=m.dev), inner, right=True).to(torch.int32).unsqueeze(0)
        return {"path": "handoff", "x": m.x(1, dim, tokens, "last"), "weight": weight, "bias": bias, "ids": ids, "cu": cu,
                "state_len": case["state_len"]}
    batch, seqlen = case["batch"], case["seqlen"]
    s = {"path": case["path"], "x": m.x(batch, dim, seqlen, case["layout"]), "weight": weight, "bias": bias,
         "ids": m.packed_ids(batch, seqlen) if case["seq_idx"] else None,
         "init": m.normal(batch, width - 1, dim).transpose(1, 2) if case["states"] else None}
    if case["path"] == "train":
        s["leaves"] = [s[k].requires_grad_() for k in ("x", "weight", "bias", "init") if s[k] is not None]
        s["grads"] = [m.x(batch, dim, seqlen, "first" if case["layout"] == "first" else "last")]
        if case["states"]:
            s["grads"].append(m.normal(batch, width - 1, dim).transpose(1, 2))
    return s


def run(s):
    if s["path"] == "decode":
        outs = [causal_conv1d_update(x, cache, weight, bias, "silu", s["lengths"], s["indices"])
                for x, cache, weight, bias in zip(s["xs"], s["caches"], s["weights"], s["biases"])]
        return {"outs": outs, "caches": s["all_caches"]}
    if s["path"] == "handoff":
        return causal_conv1d_fwd_varlen_states(s["x"], s["weight"], s["bias"], s["ids"], s["cu"], s["state_len"], "silu")
    out = causal_conv1d_fn(s["x"], s["weight"], s["bias"], seq_idx=s["ids"], initial_states=s["init"],
                           return_final_states=s["init"] is not None, activation="silu")
    if s["path"] == "prefill":
        return out
    outs = list(out) if isinstance(out, tuple) else [out]
    return {"outs": outs, "grads": torch.autograd.grad(outs, s["leaves"], s["grads"])}


def work(case):
    """Bytes: every input once and every output once per direction (a model's other layers run
    between a forward and its backward, so x is an input of both).  Operations: two per tap and
    output, three times that in the backward (the pre-activation again, dx, the sums)."""
    dim, width = case["dim"], case["width"]
    eb, wb = (4 if case[k] == "fp32" else 2 for k in ("dtype", "weights"))
    params = dim * (width + 1) * wb
    if case["path"] == "decode":
        rows = case["batch"] * (3 if case["slots"] else 4) // 4           # a quarter of the slots are padding
        if case["ring"]:
            moved = width - 1 + case["tokens"]
        else:
            moved = 2 * case["state_len"]
        per_layer = dim * eb * (rows * (moved + case["tokens"]) + case["batch"] * case["tokens"]) + params
        return {"bytes": case["layers"] * per_layer, "flops": case["layers"] * 2 * width * rows * dim * case["tokens"]}
    if case["path"] == "handoff":
        n = case["tokens"] * dim
        states = case["sequences"] * case["state_len"] * dim
        return {"bytes": (2 * n + 2 * states) * eb + 4 * case["tokens"] + params, "flops": 2 * width * n}
    n = case["batch"] * dim * case["seqlen"]
    states = case["batch"] * dim * (width - 1) if case["states"] else 0
    ids = 4 * case["batch"] * case["seqlen"] if case["seq_idx"] else 0
    forward = (2 * n + 2 * states) * eb + ids + params
    if case["path"] == "prefill":
        return {"bytes": forward, "flops": 2 * width * n}
    backward = (3 * n + 3 * states) * eb + ids + 2 * params
    return {"bytes": forward + backward, "flops": 8 * width * n}


def tolerance(case):
    return {"rel": _REL[case["dtype"]]}


def _taps(x, front, weight, bias, ids):
    """SiLU of the causal convolution of x (batch, dim, seqlen) behind `front` (batch, dim, width-1), as
    shifted products in the type of x; a tap counts where its position has the id of the output's."""
    width, seqlen = weight.shape[1], x.shape[2]
    padded = torch.cat([front, x], dim=2)
    if ids is not None:
        ids = torch.nn.functional.pad(ids, (width - 1, 0), value=-1)
    acc = bias.view(1, -1, 1).expand_as(x)
    for w in range(width):
        term = padded[:, :, w:w + seqlen] * weight[:, w].view(1, -1, 1)
        if ids is not None:
            term = torch.where((ids[:, w:w + seqlen] == ids[:, width - 1:]).unsqueeze(1), term, 0.0)
        acc = acc + term
    return acc * torch.sigmoid(acc)


def _decode_layer(x, cache, weight, bias, lengths, indices):
    width, state_len = weight.shape[1], cache.shape[2]
    new = (x.unsqueeze(2) if x.dim() == 2 else x).double()
    rows = torch.arange(new.shape[0], device=x.device) if indices is None else indices.long()
    live = rows >= 0
    old = cache[rows.clamp(min=0)]
    if lengths is None:
        window = old[:, :, state_len - (width - 1):]
        kept = torch.cat([old, new], dim=2)[:, :, -state_len:]
    else:
        at = torch.arange(-(width - 1), new.shape[2], device=x.device) + lengths.long().view(-1, 1)
        at = (at % state_len).unsqueeze(1).expand(-1, new.shape[1], -1)
        window = old.gather(2, at[..., :width - 1])
        kept = old.scatter(2, at[..., width - 1:], new)
    cache[rows[live]] = kept[live]
    out = torch.where(live.view(-1, 1, 1), _taps(new, window, weight.double(), bias.double(), None), 0.0)
    return out.squeeze(2) if x.dim() == 2 else out


def exact(case, seed):
    """What `run` returns for these inputs, in 64 bits and plain torch."""
    s = prepare(case, seed)
    if s["path"] == "decode":
        caches = s["all_caches"].double()
        outs = [_decode_layer(x, cache, weight, bias, s["lengths"], s["indices"])
                for x, cache, weight, bias in zip(s["xs"], caches.unbind(0), s["weights"], s["biases"])]
        return {"outs": outs, "caches": caches}
    leaves = [s[k].detach().double().requires_grad_(s["path"] == "train") for k in ("x", "weight", "bias")]
    x, weight, bias = leaves
    front = torch.zeros_like(x[:, :, :weight.shape[1] - 1])
    if s.get("init") is not None:
        front = s["init"].detach().double().requires_grad_(s["path"] == "train")
        leaves.append(front)
    out = _taps(x, front, weight, bias, s["ids"])
    if s["path"] == "handoff":
        n, cu = s["state_len"], s["cu"].tolist()
        states = x.new_zeros(len(cu) - 1, x.shape[1], n)
        for b, (lo, hi) in enumerate(zip(cu, cu[1:])):
            k = min(n, hi - lo)
            states[b, :, n - k:] = x[0, :, hi - k:hi]
        return out, states
    outs = [out] if s.get("init") is None else [out, x[:, :, 1 - weight.shape[1]:]]
    if s["path"] == "prefill":
        return outs[0] if len(outs) == 1 else tuple(outs)
    grads = torch.autograd.grad(outs, leaves, [g.double() for g in s["grads"]])
    return {"outs": [t.detach() for t in outs], "grads": grads}
