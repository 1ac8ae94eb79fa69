"""What the operators' Python functions refuse before anything is launched: tensors that the kernels would read or write
past the end of.  The tensors here say they are on a GPU and have no memory, so no GPU is needed, and a call that got as far
as its kernel would fail for want of an address and not with the ValueError asked for."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


@pytest.fixture(scope="module")
def ops():
    from rwkvstic_amd import ops as _ops
    return _ops


N_IN, N_OUT = 256, 48


def _product(dt):
    e = lambda n: torch.empty(n, dtype=dt, device="cuda")
    return [e(N_IN) for _ in range(3)], [torch.empty(N_IN, N_OUT, dtype=torch.uint8, device="cuda") for _ in range(3)], [e(N_OUT) for _ in range(3)], [e(N_IN) for _ in range(3)]


SHORT = {"short": lambda t: t[:-1], "expanded": lambda t: t.new_empty(1, 1).expand(1, t.numel())}


@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("how", SHORT)
@pytest.mark.parametrize("which", ["x", "y", "r"])
def test_products_of_vectors_that_are_too_short_are_refused(ops, dt, how, which):
    for i in range(3):
        with FakeTensorMode():
            x, w, y, r = _product(dt)
            t = {"x": x, "y": y, "r": r}[which]
            t[i] = SHORT[how](t[i])
            with pytest.raises(ValueError):
                ops.mm8_three(N_IN, N_OUT, *x, *w, *y, *r)
            with pytest.raises(ValueError):
                ops.mm8_one(N_IN, N_OUT, x[i], w[i], y[i], r[i])
