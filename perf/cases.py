"""What a program built on this library has it do, as cases that can be timed.

A case is a dict of plain values.  Its `kind` names the entry point:

  linear    FusedRuntime.forward: one projection, one activation (the batch-1 product of a decode step)
  group     FusedRuntime.forward_group: projections that share an activation (q/k/v, gate/up)
  sequence  FusedRuntime.plan_sequence, then FusedSequence.run: every projection group of a model as one launch
  batched   FusedRuntime.forward_batched (one projection) / forward_batched_group_into (several): M activation rows,
            as prompt processing and the verification of drafted tokens have them
  prefill   Decoder.prefill: a whole prompt through a Qwen3-architecture model
  decode    Decoder.forward_token, once per token and with its logits, over a prompt that is already in the cache

Shapes are the projections of Qwen3 4B, 8B and 14B layers.  Codes are drawn uniformly over the ball of the shell cap,
gain bits evenly, gain centroids {0.8, 1.25}, row scales exp(-4 + 0.3 g), tail columns 0.02 g, activations N(0, 1) in
binary16.  Everything is made on the GPU from the case's seed and handed over as the files' loader hands it over.
"""
import math

import numpy as np
import torch

import llvq_amd
from llvq_amd import artifact, decoder

# hidden, query heads, kv heads, intermediate (heads of 128), and the layers of the whole model
WIDTHS = {"4b": (2560, 32, 8, 9728, 36), "8b": (4096, 32, 8, 12288, 36), "14b": (5120, 40, 8, 17408, 40)}
VOCAB = 151936
HEAD_DIM = 128


def layer_groups(widths):
    """The four launch groups of a decoder layer as (d_outs, d_in): q/k/v, o, gate/up, down."""
    hidden, heads, kv, inter, _ = WIDTHS[widths]
    q, k = heads * HEAD_DIM, kv * HEAD_DIM
    return [([q, k, k], hidden), ([hidden], q), ([inter, inter], hidden), ([hidden], inter)]


def listed():
    return [
        # The smallest projection of the 4B model by itself: launch latency and the host path count.
        {"name": "linear_k_proj", "kind": "linear", "d_outs": "1024", "d_in": 2560, "cap": 12, "rotated": False, "out": "f16"},
        # An ordinary projection with f32 results (a caller that adds several projections' results up itself).
        {"name": "linear_gate_proj_f32", "kind": "linear", "d_outs": "9728", "d_in": 2560, "cap": 12, "rotated": False, "out": "f32"},
        # A projection of an artifact quantized in a rotated basis: the activation is rotated in the call.
        {"name": "linear_down_proj_rotated", "kind": "linear", "d_outs": "2560", "d_in": 9728, "cap": 12, "rotated": True, "out": "f16"},
        # The q/k/v group of a decode step.
        {"name": "group_qkv", "kind": "group", "d_outs": "4096+1024+1024", "d_in": 2560, "cap": 12, "rotated": False, "out": "f16"},
        # The largest group of a decode step, the 14B gate/up, from a cap-13 artifact (49-bit blocks in a dense stream).
        {"name": "group_gate_up_14b_cap13", "kind": "group", "d_outs": "17408+17408", "d_in": 5120, "cap": 13, "rotated": False, "out": "f16"},
        # All 252 projections of the 4B model, one token's worth, as one launch: the repository's headline workload.
        {"name": "sequence_4b", "kind": "sequence", "widths": "4b", "layers": 36, "cap": 12, "out": "f16"},
        # A handful of drafted tokens to verify, an odd number of rows.
        {"name": "batched_5_rows_f32", "kind": "batched", "d_outs": "4096", "d_in": 4096, "rotated": False, "rows": 5, "out": "f32"},
        # A speculative tree or a short prompt through a rotated artifact's q/k/v.
        {"name": "batched_qkv_64_rotated", "kind": "batched", "d_outs": "4096+1024+1024", "d_in": 4096, "rotated": True, "rows": 64, "out": "f16"},
        # A full pass of prompt rows through the widest group of an 8B layer.
        {"name": "batched_gate_up_512", "kind": "batched", "d_outs": "12288+12288", "d_in": 4096, "rotated": False, "rows": 512, "out": "f16"},
        # A prompt of a length that is no multiple of anything through a third of the 4B model.
        {"name": "prefill_4b_500", "kind": "prefill", "widths": "4b", "layers": 12, "vocab": VOCAB, "rotated": False, "kv": "f16", "head": "f16", "tokens": 500},
        # A sampling loop over the whole 4B model at a short context.
        {"name": "decode_4b", "kind": "decode", "widths": "4b", "layers": 36, "vocab": VOCAB, "rotated": False, "kv": "f16", "head": "f16", "context": 509, "tokens": 8},
        # The same at a long context with an int8 cache, int8 head and rotated artifact, on a few 14B layers.
        {"name": "decode_14b_8k_rotated", "kind": "decode", "widths": "14b", "layers": 4, "vocab": VOCAB, "rotated": True, "kv": "q8", "head": "q8", "context": 8100, "tokens": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, rotated):
    """A row length; a rotated one is an odd factor up to 31 times a power of two."""
    if not rotated:
        return _log(rng, lo, hi)
    while True:
        n = rng.choice(range(1, 32, 2)) * 2 ** rng.randrange(5, 14)
        if lo <= n <= hi:
            return n


def draw(rng):
    kind = rng.choices(("linear", "group", "sequence", "batched", "prefill", "decode"), (3, 3, 1, 3, 1, 2))[0]
    out = rng.choice(("f16", "f16", "f16", "f32"))
    rotated = rng.random() < 0.35
    if kind in ("linear", "group"):
        n = 1 if kind == "linear" else rng.randrange(2, 5)
        return {"kind": kind, "d_outs": "+".join(str(_log(rng, 64, 18000)) for _ in range(n)), "d_in": _width(rng, 200, 17408, rotated),
                "cap": 13 if rng.random() < 0.15 else 12, "rotated": rotated, "out": out}
    if kind == "sequence":
        widths = rng.choice(tuple(WIDTHS))
        return {"kind": kind, "widths": widths, "layers": _log(rng, 1, 36 if widths == "4b" else 12), "cap": 13 if rng.random() < 0.15 else 12, "out": out}
    if kind == "batched":
        n = rng.randrange(1, 4)
        return {"kind": kind, "d_outs": "+".join(str(_log(rng, 128, 13000)) for _ in range(n)), "d_in": _width(rng, 400, 13000, rotated),
                "rotated": rotated, "rows": _log(rng, 2, 600), "out": out}
    model = {"kind": kind, "widths": rng.choice(tuple(WIDTHS)), "layers": rng.randrange(1, 7), "vocab": _log(rng, 2000, 60000),
             "rotated": rotated, "kv": rng.choice(("f16", "q8")), "head": rng.choice(("f16", "q8"))}
    if kind == "prefill":
        return dict(model, tokens=_log(rng, 3, 600))
    return dict(model, context=_log(rng, 5, 8000), tokens=rng.randrange(2, 7))


# ---- inputs ------------------------------------------------------------------------
_RUNTIMES = {}


def _runtime():
    """A process has one runtime per GPU, as the matrices of all its models share the tables in it."""
    if "rt" not in _RUNTIMES:
        _RUNTIMES["rt"] = llvq_amd.FusedRuntime(device=0)
    return _RUNTIMES["rt"]


class _Maker:
    """Seeded inputs, drawn on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, dtype=torch.float32):
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).to(dtype)

    def tokens(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.gen, device="cuda").cpu().numpy().astype(np.uint32)

    def codes(self, blocks, cap):
        """The packed code stream of `blocks` blocks: 6-byte records at cap 12, 49 bits per block at cap 13."""
        top = {12: artifact.N12, 13: artifact.N13}[cap] + 1
        v = torch.randint(0, top, (blocks,), generator=self.gen, device="cuda") * 2 + torch.randint(0, 2, (blocks,), generator=self.gen, device="cuda")
        if cap == 12:
            return v.view(torch.uint8).view(-1, 8)[:, :6].flip(1).contiguous().view(-1).cpu().numpy()
        bits = (v[:, None] >> torch.arange(48, -1, -1, device="cuda")).bitwise_and_(1).to(torch.uint8).view(-1)
        bits = torch.nn.functional.pad(bits, (0, -bits.numel() % 8)).view(-1, 8)
        return (bits << torch.arange(7, -1, -1, dtype=torch.uint8, device="cuda")).sum(1, dtype=torch.uint8).cpu().numpy()

    def matrices(self, shapes, cap, rotation=None):
        """RawMatrix records of the given (name, d_out, d_in), drawn together and cut apart."""
        blocks = [d_out * (d_in // 24) for _, d_out, d_in in shapes]
        streams = [self.codes(b, cap) for b in blocks] if cap == 13 else np.split(self.codes(sum(blocks), cap), np.cumsum(blocks)[:-1] * 6)
        scales = torch.exp(-4.0 + 0.3 * self.normal(sum(s[1] for s in shapes)).double()).cpu().numpy()
        tails = [d_out * (d_in % 24) for _, d_out, d_in in shapes]
        tail = (0.02 * self.normal(sum(tails))).cpu().numpy()
        scales, tail = np.split(scales, np.cumsum([s[1] for s in shapes])[:-1]), np.split(tail, np.cumsum(tails)[:-1])
        return [artifact.RawMatrix(n, do, di, cap, (0.8, 1.25), s, t, c, rotation_seed=rotation)
                for (n, do, di), s, t, c in zip(shapes, scales, tail, streams)]


class _Products:
    """Uploaded projections and what their calls take; the device memory is given back with the object."""

    def __init__(self):
        self.rt, self.projs, self.seq = _runtime(), [], None

    def upload(self, raws):
        got = [self.rt.upload(r) for r in raws]
        self.projs += got
        return got

    def __del__(self):
        if self.seq is not None:
            self.seq.close()
        for p in self.projs:
            self.rt.free(p)


def _dtype(case):
    return torch.float16 if case["out"] == "f16" else torch.float32


def _prepare_products(case, make):
    s = _Products()
    s.case, s.dtype = case, _dtype(case)
    if case["kind"] == "sequence":
        groups, ys = [], 0
        for layer in range(case["layers"]):
            for g, (d_outs, d_in) in enumerate(layer_groups(case["widths"])):
                groups.append((s.upload(make.matrices([("model.layers.%d.g%d.p%d.weight" % (layer, g, j), d, d_in) for j, d in enumerate(d_outs)], case["cap"])), d_in))
                ys += sum(d_outs)
        xs = {d_in: make.normal(d_in, dtype=torch.float16) for _, d_in in layer_groups(case["widths"])}
        s.y = torch.empty(ys, dtype=s.dtype, device="cuda")
        items, at = [], 0
        for projs, d_in in groups:
            outs = []
            for p in projs:
                outs.append(s.y[at:at + p.d_out])
                at += p.d_out
            items.append((projs, xs[d_in], False, outs))
        s.seq = s.rt.plan_sequence(items, out_dtype=s.dtype)
        return s
    shapes = [("model.layers.0.p%d.weight" % j, int(d), case["d_in"]) for j, d in enumerate(case["d_outs"].split("+"))]
    projs = s.upload(make.matrices(shapes, case.get("cap", 12), 0x5EED if case["rotated"] else None))
    if case["kind"] == "batched":
        s.x = make.normal(case["rows"], case["d_in"], dtype=torch.float16)
        s.rt.reserve_batched(projs, case["rows"])
        if len(projs) > 1:
            s.ys = [torch.empty((case["rows"], p.d_out), dtype=s.dtype, device="cuda") for p in projs]
    else:
        s.x = make.normal(case["d_in"], dtype=torch.float16)
    return s


def _table(make, vocab, hidden, kind):
    if kind == "f16":
        return make.normal(vocab, hidden, dtype=torch.float16).cpu().numpy()
    codes = torch.randint(0, 256, (vocab * hidden,), generator=make.gen, device="cuda", dtype=torch.uint8)
    scales = (0.02 + 0.002 * torch.rand(vocab * hidden // 64, generator=make.gen, device="cuda")).half()
    biases = (-127.5 * scales.float()).half()
    return artifact.RawTensor("model.embed_tokens.weight", [vocab, hidden], bits=8, group=64, packed=codes.cpu().numpy(),
                              scales=scales.view(torch.int16).cpu().numpy().view(np.uint16), biases=biases.view(torch.int16).cpu().numpy().view(np.uint16))


class _Model:
    pass


def _prepare_model(case, make):
    hidden, heads, kv, inter, _ = WIDTHS[case["widths"]]
    prompt, steps = (0, case["tokens"]) if case["kind"] == "prefill" else (case["context"], case["tokens"])
    cfg = decoder.Qwen3Config(case["layers"], hidden, heads, kv, HEAD_DIM, inter, case["vocab"], max_positions=prompt + steps,
                              tie_word_embeddings=True, kv_mode=case["kv"])
    layers = [make.matrices([("model.layers.%d.%s.weight" % (i, site), do, di) for site, do, di in cfg.shapes()], 12, 0x5EED if case["rotated"] else None)
              for i in range(case["layers"])]

    def gains(*shape):
        return (1.0 + 0.1 * make.normal(*shape)).half().cpu().numpy()

    n = case["layers"]
    weights = decoder.DecoderWeights(gains(n, hidden), gains(n, hidden), gains(n, HEAD_DIM), gains(n, HEAD_DIM), gains(hidden),
                                     _table(make, case["vocab"], hidden, case["head"]))
    s = _Model()
    s.case, s.context = case, prompt
    s.dec = decoder.Decoder(_runtime(), cfg, layers, weights, prefill_rows=512)
    s.tokens = make.tokens(steps, case["vocab"])
    if prompt:
        s.dec.prefill(make.tokens(prompt, case["vocab"]), want_logits=False)
    return s


def prepare(case, seed):
    make = _Maker(seed)
    return _prepare_model(case, make) if case["kind"] in ("prefill", "decode") else _prepare_products(case, make)


def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "linear":
        return state.rt.forward(state.projs[0], state.x, out_dtype=state.dtype)
    if kind == "group":
        return state.rt.forward_group(state.projs, state.x, out_dtype=state.dtype)
    if kind == "sequence":
        state.seq.run()
        return state.y
    if kind == "batched":
        if len(state.projs) > 1:
            return state.rt.forward_batched_group_into(state.projs, state.x, state.ys)
        return state.rt.forward_batched(state.projs[0], state.x, out_dtype=state.dtype)
    if kind == "prefill":
        state.dec.reset()
        return state.dec.prefill(state.tokens)[0]
    # back to the end of the prompt, whose keys and values are in the cache, then one token at a time
    state.dec.seek(state.context)
    return [state.dec.forward_token(t)[0] for t in state.tokens]


# ---- what a pass cannot do without ---------------------------------------------------
def _matrix_bytes(d_out, d_in, cap):
    blocks = d_out * (d_in // 24)
    return (blocks * (48 if cap == 12 else 49) + 7) // 8 + 4 * d_out * (d_in % 24) + 4 * d_out


def work(case):
    kind = case["kind"]
    if kind in ("linear", "group", "batched"):
        rows, d_in, width = case.get("rows", 1), case["d_in"], 2 if case["out"] == "f16" else 4
        d_outs = [int(d) for d in case["d_outs"].split("+")]
        return {"bytes": sum(_matrix_bytes(d, d_in, case.get("cap", 12)) + width * rows * d for d in d_outs) + 2 * rows * d_in,
                "flops": 2.0 * rows * d_in * sum(d_outs)}
    groups = layer_groups(case["widths"])
    weights = case["layers"] * sum(_matrix_bytes(d, d_in, case.get("cap", 12)) for ds, d_in in groups for d in ds)
    macs = case["layers"] * sum(d * d_in for ds, d_in in groups for d in ds)
    if kind == "sequence":
        width = 2 if case["out"] == "f16" else 4
        return {"bytes": weights + case["layers"] * width * sum(sum(ds) for ds, _ in groups) + 2 * sum({d_in for _, d_in in groups}), "flops": 2.0 * macs}
    hidden, heads, kv, _, _ = WIDTHS[case["widths"]]
    row = 2 * kv * HEAD_DIM * (2 if case["kv"] == "f16" else 1 + 4 / 64)  # a position's keys and values
    head = case["vocab"] * hidden * (2 if case["head"] == "f16" else 1 + 4 / 64)
    n = case["tokens"]
    if kind == "prefill":  # weights once, cache rows written, the head on the last position
        return {"bytes": weights + head + case["layers"] * n * row + 4 * case["vocab"],
                "flops": 2.0 * macs * n + 2.0 * case["vocab"] * hidden + case["layers"] * 2.0 * heads * HEAD_DIM * n * (n + 1)}
    seen = sum(case["context"] + t + 1 for t in range(n))  # cache rows read over the steps: weights and head once per step
    return {"bytes": n * (weights + head + 4 * case["vocab"]) + case["layers"] * seen * row,
            "flops": n * 2.0 * (macs + case["vocab"] * hidden) + case["layers"] * 4.0 * heads * HEAD_DIM * seen}


def tolerance(case):
    if case["kind"] in ("prefill", "decode"):
        return {"rel": 1e-2}  # binary16 activations through every layer
    if case["kind"] == "batched":
        return {"rel": 1e-3}  # weights are binary16 operands of the matrix cores
    return {"rel": 1e-3} if case["out"] == "f16" else {"rel": 1e-5}
