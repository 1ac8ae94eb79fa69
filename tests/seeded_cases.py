"""Recipes behind tests/golden/seeded.json: seeded draws, token steps, prompts and replies, as whole numbers or digests of
bits.  The recorded values were written by running these functions on the library as it was before its prompts, its
sampler and its quantiser were first made faster: a program that seeds its generator keeps its texts across versions, and
one draw that rounding tips over changes every token after it.  (``python tests/seeded_cases.py draws ... > out.json``.)"""
import hashlib
import json
import os
import sys

import torch

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "seeded.json")


def _digest(*tensors):
    h = hashlib.sha256()
    for t in tensors:
        h.update(t.detach().cpu().contiguous().numpy().tobytes())
    return h.hexdigest()[:16]


def draws():
    """Tokens chosen by the typical sampler: 100 distributions, 48 draws of each."""
    from rwkvstic_amd import ops
    out = {}
    for i in range(240, 340):
        g = torch.Generator().manual_seed(1000 + i)
        spread, tau, temp = ((0.6, 0.8, 1.0), (1.0, 0.95, 0.7), (2.5, 0.8, 1.0), (0.3, 0.5, 1.0))[i % 4]
        logits = (torch.randn(50277, generator=g, dtype=torch.float64) * spread).cuda()
        toks = torch.empty(48, dtype=torch.int64, device="cuda")
        for k in range(48):
            ops.sample_token(logits, temp=temp, tau=tau, seed=77, counter=k, out=toks[k:k + 1])
        out[str(i)] = _digest(toks)
    return out


def edge_draws():
    """Tokens chosen by the typical sampler from distributions of other shapes, vocabularies on both sides of the 8192 from
    which logits are loaded in pairs, and cuts from a few tokens to all of them.  (Recorded from the sampler that
    searched the cut bit by bit in passes over all tokens.)"""
    from rwkvstic_amd import ops
    out = {}
    for V in (300, 8191, 8192, 8193, 20001, 50277, 53247, 53248):
        for shape in ("normal", "zipf", "peaked", "masked", "equal"):
            x = torch.randn(V, generator=torch.Generator().manual_seed(V), dtype=torch.float64) * 1.5
            if shape == "zipf":
                x = -1.3 * torch.log(torch.arange(1, V + 1, dtype=torch.float64))
            elif shape == "peaked":
                x[V - 1] += 14.0
                x[3] += 16.0
            elif shape == "masked":
                x[: V // 2] = -float("inf")
            elif shape == "equal":
                x = x * 0 + 0.25
            logits = x.cuda()
            for tau, temp in ((0.2, 1.0), (0.8, 1.0), (0.95, 0.7), (0.99999, 1.3), (1.0, 1.0), (1.5, 1.0)):
                toks = torch.empty(24, dtype=torch.int64, device="cuda")
                for k in range(24):
                    ops.sample_token(logits, temp=temp, tau=tau, seed=V, counter=k, out=toks[k:k + 1])
                out[f"{V} {shape} {tau} {temp}"] = _digest(toks)
    return out


def _models():
    """Models made of random codes, so that no quantiser has a part in them: (name, model)."""
    from rwkvstic_amd.model import HipRWKV
    for L, C, V in ((2, 1024, 1000), (2, 2560, 1000), (1, 5120, 1000)):
        g = torch.Generator().manual_seed(C)
        F = 4 * C

        def u(*shape, lo=0.0, hi=1.0, dtype=torch.float64):
            return (torch.rand(*shape, generator=g) * (hi - lo) + lo).to(dtype)

        tree = {"emb.w": u(V, C, lo=-0.04, hi=0.04, dtype=torch.float32)}

        def mat(prefix, suffix, n_in, n_out):
            tree[f"{prefix}weight{suffix}"] = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8)
            tree[f"{prefix}range{suffix}"] = u(n_in, lo=2e-4, hi=6e-4, dtype=torch.float32)
            tree[f"{prefix}offset{suffix}"] = u(n_in, lo=-0.06, hi=-0.04)

        for ln in ("ln_in", "ln_out") + tuple(f"blocks.{i}.ln{k}" for i in range(L) for k in (1, 2)):
            tree[ln + ".weight"], tree[ln + ".bias"] = u(C, lo=0.5, hi=1.5), u(C, lo=-0.1, hi=0.1)
        mat("head.weights.0.", "", C, V)
        for i in range(L):
            p = f"blocks.{i}."
            tree[p + "attmix"], tree[p + "ffnmix"] = u(3, 1, C), u(2, 1, C)
            tree[p + "time_first"], tree[p + "time_decay"] = u(C, lo=-1.0), -torch.exp(u(C, lo=-5.0))
            for s in ("", "1", "2"):
                mat(p + "att.weights.0.", s, C, C)
            mat(p + "attout.weights.0.", "", C, C)
            mat(p + "ffnkey.weights.0.", "", C, F)
            mat(p + "ffnreceptance.weights.0.", "", C, C)
            mat(p + "ffnvalue.weights.0.", "", F, C)
        yield str(C), HipRWKV.from_quantized(tree)


def _tokens(n, seed):
    return torch.randint(0, 1000, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def steps():
    """Logits and state after token steps, one by one."""
    out = {}
    for name, m in _models():
        st = m.emptyState.clone()
        for i, t in enumerate(_tokens(6, 1)):
            lg, st = m.forward([t], st)
            out[f"{name} step {i}"] = _digest(lg, st)
    return out


def prompts():
    """Logits and state after prompts of every path's lengths, from a state that is not empty."""
    out = {}
    for name, m in _models():
        _, start = m.forward(_tokens(3, 2), m.emptyState.clone())
        for T in (4, 5, 6, 8, 9, 24, 32, 33, 63, 64, 65, 77, 127, 128, 300, 513, 1030):
            lg, st = m.forward(_tokens(T, T), start.clone())
            out[f"{name} prompt {T}"] = _digest(lg, st)
    return out


def replies():
    """Sampled answers to prompts, from a checkpoint that is quantised here: 24 layers of 1024 channels."""
    from rwkvstic_amd import synth
    from rwkvstic_amd.master import RWKVMaster, typical
    from rwkvstic_amd.model import HipRWKV
    m = HipRWKV(synth.iter_tensors(24, 1024, 4096, 50277, seed=11, device="cuda", ln="random"))
    ma = RWKVMaster(m, m.emptyState, typical)
    out = {}
    for s in range(40):
        torch.manual_seed(s)
        ma.resetState()
        ma.loadContext(newctx=synth.random_tokens(77 if s % 2 else 3 + s, seed=s).tolist())
        out[str(s)] = ma.encode(ma.forward(number=24)["output"])
    return out


if __name__ == "__main__":
    sys.path.insert(0, os.getcwd())
    print(json.dumps({name: globals()[name]() for name in sys.argv[1:]}))
