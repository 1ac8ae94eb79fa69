"""The work a user of this framework has it do, as cases that can be timed and compared.

Kinds of case (the key ``"kind"``), each through the public entry points of ``rwkvstic_amd``:

``tokens``     a generation loop on the device: ``HipRWKV.decode_greedy`` / ``decode_sample`` at batch 1.
``chat``       one turn of a conversation: ``RWKVMaster.loadContext`` of a prompt, then ``forward(number=n)``.
``prompt``     ``HipRWKV.forward`` of a whole prompt (or one chunk of it): state and next-token logits.
``batch``      ``HipRWKV.forward_batch``: one token for each of B independent sequences.
``products``   the quantised matrix-vector products on their own, 1..8 vectors, in either packed layout.
``wkv``        the float32 WKV recurrence on its own.
``operators``  the three drop-in operators ``torch.ops.rwkv.*`` as a reference-style layer calls them: the float64
               recurrence over a prompt chunk, then the recurrence and the products of one more token.
``load``       quantising and packing the seven matrices of a layer of a float32 checkpoint.

Models are random-init checkpoints (``rwkvstic_amd.synth``) with LayerNorm parameters that are not the identity, so that
every weight and bias path carries a value.
"""
from __future__ import annotations

import math

import torch

from rwkvstic_amd import ops, synth
from rwkvstic_amd.master import RWKVMaster, greedy, typical
from rwkvstic_amd.model import HipRWKV, QuantMatrix

VOCAB = 50277

# Widths of the model family (ffn width = 4 x), and two in between that a model trained at home might have.
WIDTHS = (512, 768, 1024, 1536, 2048, 2560, 4096, 5120)
# Widths whose sampled generation runs on the device (``decode_sample``); the others sample on the host.
DEVICE_LOOP_WIDTHS = (1024, 2048, 2560, 4096, 5120)


def listed():
    return [
        # The smallest model of the family: a token is 124 MB of weights, so latency and launches decide.
        dict(name="tokens-169M", kind="tokens", layers=12, width=768, vocab=VOCAB, n=32, pick="greedy"),
        # The headline workload: batch-1 greedy decode of the 3B shape.
        dict(name="tokens-3B", kind="tokens", layers=32, width=2560, vocab=VOCAB, n=16, pick="greedy"),
        # The largest shape at batch 1, with the sampler the loader installs by default.
        dict(name="tokens-14B", kind="tokens", layers=40, width=5120, vocab=VOCAB, n=4, pick="typical"),
        # A conversation turn with a small model: a short prompt of odd length, then a short answer.
        dict(name="chat-1024", kind="chat", layers=24, width=1024, vocab=VOCAB, prompt=77, n=24, pick="typical"),
        # Reading a document: the 1024-token prompt of the headline workload.
        dict(name="prompt-3B", kind="prompt", layers=32, width=2560, vocab=VOCAB, tokens=1024),
        # The largest shape's prompt chunk.
        dict(name="prompt-14B", kind="prompt", layers=40, width=5120, vocab=VOCAB, tokens=256),
        # Serving a few users at once ...
        dict(name="batch-3B", kind="batch", layers=32, width=2560, vocab=VOCAB, batch=8),
        # ... and serving many with the largest shape.
        dict(name="batch-14B", kind="batch", layers=40, width=5120, vocab=VOCAB, batch=32),
        # The 3B shape's three matrix shapes, eight vectors each.
        dict(name="products-3B", kind="products", width=2560, batch=8, layout="m16"),
        # The recurrence alone over a batch of long sequences.
        dict(name="wkv-f32", kind="wkv", batch=8, tokens=1024, width=2560),
        # A reference-style model on the drop-in operators: a prompt chunk, then one token.
        dict(name="operators-3B", kind="operators", width=2560, tokens=256),
        # Loading a checkpoint: one layer of the 3B shape.
        dict(name="load-3B", kind="load", width=2560),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of lo..hi."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _model(rng, widths=WIDTHS):
    """Layers, width and vocabulary of a model no larger than the largest listed one."""
    width = rng.choice(widths)
    # (5 to 40 layers' worth of depth; the family pairs 12 with the smallest width and 40 with the largest)
    layers = min(40, max(2, _log(rng, 4, 40)))
    vocab = VOCAB if rng.random() < 0.7 else _log(rng, 4000, 50000)
    return dict(layers=layers, width=width, vocab=vocab)


def draw(rng):
    kind = rng.choice(("tokens", "tokens", "chat", "prompt", "prompt", "batch", "batch", "products", "wkv", "operators", "load"))
    case = dict(kind=kind)
    if kind == "tokens":
        case.update(_model(rng))
        case["n"] = _log(rng, 1, 32)
        if case["layers"] * case["width"] ** 2 * case["n"] > 4 * 40 * 5120 ** 2:
            case["n"] = 4
        case["pick"] = "typical" if case["width"] in DEVICE_LOOP_WIDTHS and rng.random() < 0.4 else "greedy"
    elif kind == "chat":
        case.update(_model(rng, (768, 1024, 2048, 2560)))
        case["prompt"] = _log(rng, 1, 512)
        case["n"] = _log(rng, 1, 24)
        case["pick"] = "typical" if case["width"] in DEVICE_LOOP_WIDTHS else "greedy"
    elif kind == "prompt":
        case.update(_model(rng))
        case["tokens"] = _log(rng, 2, 2048)
        # (no more than the largest listed prompt)
        most = 256 * 40 * 5120 ** 2 / (case["layers"] * case["width"] ** 2)
        case["tokens"] = max(2, min(case["tokens"], int(most)))
    elif kind == "batch":
        case.update(_model(rng))
        case["batch"] = _log(rng, 1, 160)
        if case["layers"] * case["width"] ** 2 > 20 * 5120 ** 2:
            case["batch"] = min(case["batch"], 32)
    elif kind == "products":
        case["width"] = 64 * rng.randint(8, 64)
        case["layout"] = rng.choice(("m16", "packed"))
        case["batch"] = rng.randint(1, 8) if case["layout"] == "m16" else rng.choice((1, 2, 4, 8))
    elif kind == "wkv":
        case["width"] = rng.choice(WIDTHS) + rng.choice((0, 0, 0, 3, 40))
        case["tokens"] = _log(rng, 1, 2048)
        case["batch"] = max(1, min(_log(rng, 1, 16), 8 * 1024 * 2560 // (case["tokens"] * case["width"])))
    elif kind == "operators":
        case["width"] = rng.choice(WIDTHS) + rng.choice((0, 0, 8, 24))
        case["tokens"] = _log(rng, 1, 1024)
    else:
        case["width"] = 64 * rng.randint(8, 48)
    return case


# ---------------------------------------------------------------- inputs
class _State:
    pass


def _build(case, seed):
    w = case["width"]
    return HipRWKV(synth.iter_tensors(case["layers"], w, 4 * w, case["vocab"], seed=seed, device="cuda", ln="random"), device="cuda:0")


def _product_shapes(width):
    return (width, width), (width, 4 * width), (4 * width, width)


def _codes(g, n_in, n_out):
    return torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8, device="cuda")


def _rand(g, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
    return (torch.rand(*shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo).to(dtype)


def _randn(g, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * scale).to(dtype)


def prepare(case, seed):
    s = _State()
    s.case, s.seed, kind, w = case, seed, case["kind"], case["width"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + 17)
    if kind in ("tokens", "chat", "prompt", "batch"):
        s.model = _build(case, seed)
        ids = synth.random_tokens(4096, V=case["vocab"], seed=seed)
        if kind == "chat":
            s.master = RWKVMaster(s.model, s.model.emptyState, typical if case["pick"] == "typical" else greedy)
            s.prompt = ids[:case["prompt"]].tolist()
        elif kind == "batch":
            # sequences that have each read a few tokens of their own
            b = case["batch"]
            s.states = s.model.emptyState.repeat(b, 1, 1, 1).contiguous()
            for i in range(3):
                _, s.states = s.model.forward_batch(ids[i * b:(i + 1) * b].cuda(), s.states)
            s.tokens = ids[3 * b:4 * b].cuda()
        else:
            # what came before: a short prompt
            _, s.state = s.model.forward(ids[:24].cuda(), s.model.emptyState.clone())
            s.token = int(ids[24])
            s.tokens = ids[25:25 + case.get("tokens", 0)].cuda()
    elif kind == "products":
        s.mats = []
        for n_in, n_out in _product_shapes(w):
            codes = _codes(g, n_in, n_out)
            packed = ops.pack_m16(codes) if case["layout"] == "m16" else ops.pack(codes)
            s.mats.append((_randn(g, case["batch"], n_in), packed, n_in, n_out,
                           _rand(g, n_in, lo=1e-4, hi=1e-3), _randn(g, n_in, scale=0.01, dtype=torch.float64),
                           _rand(g, n_out, lo=1e-4, hi=1e-3), _randn(g, n_out, scale=0.01)))
    elif kind == "wkv":
        b, t = case["batch"], case["tokens"]
        s.k, s.v = _randn(g, b, t, w), _randn(g, b, t, w)
        s.w, s.u = -torch.exp(_rand(g, w, lo=-8.0, hi=1.0)), _rand(g, w, lo=-1.0, hi=1.0)
    elif kind == "operators":
        ops.register_torch_ops()
        t, f64 = case["tokens"], torch.float64
        # the three matrices that share an input, the att output, ffn key, ffn receptance and ffn value
        s.three = [(_randn(g, w), _codes(g, w, w), _rand(g, w, lo=1e-4, hi=1e-3)) for _ in range(3)]
        s.ones = [(n_in, n_out, _randn(g, n_in), _codes(g, n_in, n_out), _rand(g, n_in, lo=1e-4, hi=1e-3))
                  for n_in, n_out in ((w, w), (w, 4 * w), (w, w), (4 * w, w))]
        s.k, s.v = _randn(g, t, w, dtype=f64), _randn(g, t, w, dtype=f64)
        s.k1, s.v1 = _randn(g, 1, w, dtype=f64), _randn(g, 1, w, dtype=f64)
        s.w, s.u = -torch.exp(_rand(g, w, lo=-5.0, hi=1.0, dtype=f64)), _rand(g, w, lo=-1.0, hi=1.0, dtype=f64)
        s.aa, s.bb = _randn(g, w, dtype=f64), _rand(g, w, lo=0.5, hi=2.0, dtype=f64)
    else:
        s.weights = [_randn(g, n_out, n_in, scale=0.02)
                     for n_in, n_out in ((w, w), (w, w), (w, w), (w, w), (w, 4 * w), (w, w), (4 * w, w))]
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "tokens":
        state = s.state.clone()
        if case["pick"] == "greedy":
            toks, logits, state = s.model.decode_greedy(s.token, case["n"], state)
        else:
            toks, logits, state = s.model.decode_sample(s.token, case["n"], state, end_adj=-990.0, seed=s.seed)
        return {"tokens": toks, "logits": logits, "state": state}
    if kind == "chat":
        torch.manual_seed(s.seed)               # the sampler's seed is drawn from torch's generator
        s.master.resetState()
        s.master.loadContext(newctx=s.prompt)
        reply = s.master.forward(number=case["n"])
        return {"tokens": torch.tensor(s.master.encode(reply["output"])), "logits": reply["logits"], "state": reply["state"]}
    if kind == "prompt":
        logits, state = s.model.forward(s.tokens, s.state.clone())
        return {"logits": logits, "state": state}
    if kind == "batch":
        logits, states = s.model.forward_batch(s.tokens, s.states.clone())
        return {"logits": logits, "states": states}
    if kind == "products":
        fn = ops.mm8_m16 if case["layout"] == "m16" else ops.mm8_packed
        return [fn(x, packed, n_in, n_out, r_row, m_row, r_col, m_col)
                for x, packed, n_in, n_out, r_row, m_row, r_col, m_col in s.mats]
    if kind == "wkv":
        b, w = case["batch"], case["width"]
        aa, bb = torch.zeros(b, w, device="cuda"), torch.zeros(b, w, device="cuda")
        pp = torch.full((b, w), -1e38, device="cuda")
        return [ops.wkv_f32(s.w, s.u, s.k, s.v, aa, bb, pp), aa, bb, pp]
    if kind == "operators":
        w, t, rwkv = case["width"], case["tokens"], torch.ops.rwkv
        aa, bb, pp = s.aa.clone(), s.bb.clone(), torch.zeros_like(s.aa)
        y = torch.empty_like(s.k)
        rwkv.wkv_forward(1, t, w, s.w, s.u, s.k, s.v, y, aa, bb, pp)
        out = torch.zeros(3, w, device="cuda")
        (x0, w0, r0), (x1, w1, r1), (x2, w2, r2) = s.three
        rwkv.mm8_three(w, w, x0, x1, x2, w0, w1, w2, out[0], out[1], out[2], r0, r1, r2)
        y1 = torch.empty_like(s.k1)
        rwkv.wkv_forward(1, 1, w, s.w, s.u, s.k1, s.v1, y1, aa, bb, pp)
        outs = [y, y1, aa, bb, out]
        for n_in, n_out, x, codes, r in s.ones:
            o = torch.zeros(n_out, device="cuda")
            rwkv.mm8_one(n_in, n_out, x, codes, o, r)
            outs.append(o)
        return outs
    mats = [QuantMatrix.from_weight(x, x.device) for x in s.weights]
    return [(m.packed, m.packed16, m.range, m.offset) for m in mats]


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind, w = case["kind"], case["width"]
    if kind in ("tokens", "chat", "prompt", "batch"):
        body, head = case["layers"] * 13 * w * w, case["vocab"] * w
        state = 2 * case["layers"] * 5 * w * 8
        token = dict(bytes=body + head + 4 * w + state + 8 * case["vocab"], flops=2 * (body + head))
        if kind == "tokens":
            return {k: case["n"] * v for k, v in token.items()}
        if kind == "batch":
            b = case["batch"]
            return {"bytes": body + head + b * (4 * w + state + 8 * case["vocab"]), "flops": b * 2 * (body + head)}
        t = case["tokens"] if kind == "prompt" else case["prompt"]
        prompt = {"bytes": token["bytes"] + (t - 1) * 4 * w, "flops": 2 * (t * body + head)}
        if kind == "prompt":
            return prompt
        return {k: prompt[k] + case["n"] * token[k] for k in token}
    if kind == "products":
        b = case["batch"]
        return {"bytes": sum(i * o + b * (4 * i + 8 * o) + 12 * i + 8 * o for i, o in _product_shapes(w)),
                "flops": sum(2 * b * i * o for i, o in _product_shapes(w))}
    if kind == "wkv":
        n = case["batch"] * case["tokens"] * w
        return {"bytes": 12 * n + 24 * case["batch"] * w + 8 * w, "flops": 16 * n}
    if kind == "operators":
        n = (case["tokens"] + 1) * w
        return {"bytes": 24 * n + 48 * w + 13 * w * w + 4 * 4 * 17 * w, "flops": 8 * n + 2 * 13 * w * w}
    return {"bytes": 13 * w * w * 6 + 12 * 10 * w, "flops": 13 * w * w * 4}


def tolerance(case):
    """About four times the distance between two correct orders of the same sums, as measured on these cases."""
    kind = case["kind"]
    if kind in ("tokens", "chat", "prompt", "batch"):
        # one prompt token by token, in chunks and whole: 4e-7, largest single value 1.9e-6
        return {"rel": 2e-6, "max": 2e-5}
    if kind == "products":
        # against float64: 3e-12 with exact integer sums, 2e-9 with float32 chains (the zero-point terms, which are
        # float64 in both, are most of the result)
        return {"rel": 2e-11} if case["layout"] == "m16" else {"rel": 1e-8}
    if kind == "wkv":
        # against float64: 1.5e-7, largest single value 2e-6
        return {"rel": 6e-7, "max": 1e-5}
    if kind == "operators":
        # the float32 products against float64: 2.5e-7 (the float64 recurrence: 5e-16)
        return {"rel": 1e-6}
    # codes are whole numbers and stay the same; ranges and offsets are float sums over a column
    return {"rel": 1e-14}
