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


if __name__ == "__main__":
    sys.path.insert(0, os.getcwd())
    print(json.dumps({name: globals()[name]() for name in sys.argv[1:]}))
