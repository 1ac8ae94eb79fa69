"""The operators without their native host side (not built, or built for another torch): the same kernels, through Python."""
import os
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import sys, warnings
import torch
sys.modules["rwkvstic_amd._rwkv_torch"] = None            # importing it fails
from rwkvstic_amd import ops
with warnings.catch_warnings(record=True) as said:
    warnings.simplefilter("always")
    ops.register_torch_ops()
assert any("_rwkv_torch.so" in str(w.message) for w in said)
print(*(str(getattr(torch.ops.rwkv, n).default._schema) for n in ("wkv_forward", "mm8_one", "mm8_three")), sep="\\n")
try:
    ops.mm8_packed(torch.zeros(1, 4), None, 4, 4, None, None)
except ValueError as e:
    print(e)
"""


def test_operators_are_published_and_called_without_it():
    run = lambda program: subprocess.run([sys.executable, "-c", program], cwd=ROOT, capture_output=True, text=True, check=True).stdout.splitlines()
    without = run(PROGRAM)
    assert without[3] == "x must be a CUDA tensor"
    assert without[:3] == run(PROGRAM.replace('sys.modules["rwkvstic_amd._rwkv_torch"] = None', "").replace("assert any", "assert not any"))[:3]


@pytest.mark.gpu
def test_results_are_the_same_without_it(monkeypatch):
    from rwkvstic_amd import _native as N, ops
    g = torch.Generator().manual_seed(3)
    n_in, n_out = 192, 100
    codes = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8).cuda()
    x, r, m = torch.randn(4, n_in, generator=g).cuda(), torch.rand(n_in, generator=g).cuda(), torch.randn(n_in, generator=g).double().cuda()
    f = lambda *s: torch.rand(*s, generator=g).cuda()
    wkv = -f(40), f(40), f(2, 7, 40), f(2, 7, 40), f(2, 40), f(2, 40) + 0.5, f(2, 40)

    def results():
        state = [t.clone() for t in wkv[4:]]
        return [ops.mm8_packed(x, ops.pack(codes), n_in, n_out, r, m), ops.mm8_m16(x, ops.pack_m16(codes), n_in, n_out, r, m),
                ops.wkv_f32(*wkv[:4], *state), *state]

    want = results()
    monkeypatch.setattr(N, "_host", (N.lib(), None))
    assert all(torch.equal(a, b) for a, b in zip(want, results()))
