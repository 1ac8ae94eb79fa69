"""What the operators refuse before anything is launched: tensors that the kernels would read or write past the end of.
Without a GPU the tensors say they are on one and have no memory: the Python functions look at them, and a call that got as
far as its kernel would fail for want of an address and not with the ValueError asked for.  On a GPU the native side looks first."""
from contextlib import nullcontext

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


ON = pytest.mark.parametrize("tensors", [pytest.param(FakeTensorMode, id="no GPU"), pytest.param(nullcontext, id="GPU", marks=pytest.mark.gpu)])


@pytest.fixture(scope="module")
def ops():
    from rwkvstic_amd import ops as _ops
    return _ops


N_IN, N_OUT = 256, 48


def _product(dt):
    e = lambda n: torch.empty(n, dtype=dt, device="cuda")
    return [e(N_IN) for _ in range(3)], [torch.empty(N_IN, N_OUT, dtype=torch.uint8, device="cuda") for _ in range(3)], [e(N_OUT) for _ in range(3)], [e(N_IN) for _ in range(3)]


SHORT = {"short": lambda t: t[:-1], "expanded": lambda t: t.new_empty(1, 1).expand(1, t.numel())}


@ON
@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("how", SHORT)
@pytest.mark.parametrize("which", ["x", "y", "r"])
def test_products_of_vectors_that_are_too_short_are_refused(ops, tensors, dt, how, which):
    for i in range(3):
        with tensors():
            x, w, y, r = _product(dt)
            t = {"x": x, "y": y, "r": r}[which]
            t[i] = SHORT[how](t[i])
            with pytest.raises(ValueError):
                ops.mm8_three(N_IN, N_OUT, *x, *w, *y, *r)
            with pytest.raises(ValueError):
                ops.mm8_one(N_IN, N_OUT, x[i], w[i], y[i], r[i])


def _matvec(ops, layout):
    """A product of 4 vectors that fits: its arguments by name."""
    e = lambda *s, dtype=torch.float32: torch.empty(*s, dtype=dtype, device="cuda")
    n = (ops.N.lib().rwkv_packed_bytes if layout == "packed" else ops.N.lib().rwkv_packed_m16_bytes)(N_IN, N_OUT)
    return dict(x=e(4, N_IN), packed=e(n, dtype=torch.uint8), r_row=e(N_IN), m_row=e(N_IN, dtype=torch.float64), r_col=e(N_OUT), m_col=e(N_OUT),
                out=e(4, N_OUT, dtype=torch.float64), workspace=e(1 << 20, dtype=torch.uint8))


def _strided(t):
    return torch.stack((t, t), -1)[..., 0]


WRONG = {"short": lambda t: t.reshape(-1)[:-1], "strided": _strided, "on the host": lambda t: torch.empty(t.shape, dtype=t.dtype, device="cpu")}


@ON
@pytest.mark.parametrize("layout,which,how", [(layout, which, how) for layout in ("packed", "m16") for which in ("packed", "r_row", "m_row", "r_col", "m_col", "out")
                                              for how in WRONG] + [("m16", "workspace", "strided"), ("m16", "workspace", "on the host")])
def test_matvec_buffers_that_do_not_hold_the_product_are_refused(ops, tensors, layout, which, how):
    with tensors():
        a = _matvec(ops, layout)
        a[which] = WRONG[how](a[which])
        ws = {"workspace": a["workspace"]} if layout == "m16" else {}
        with pytest.raises(ValueError):
            (ops.mm8_packed if layout == "packed" else ops.mm8_m16)(a["x"], a["packed"], N_IN, N_OUT, a["r_row"], a["m_row"], a["r_col"], a["m_col"], out=a["out"], **ws)


@ON
@pytest.mark.parametrize("out", [dict(size=(1,), dtype=torch.int64, device="cpu"), dict(size=(1,), dtype=torch.int32, device="cuda"), dict(size=(0,), dtype=torch.int64, device="cuda")])
def test_tokens_go_nowhere_but_to_a_word_of_the_device(ops, tensors, out):
    with tensors():
        logits, out = torch.empty(64, dtype=torch.float64, device="cuda"), torch.empty(**out)
        for call in (ops.argmax, ops.sample_token):
            with pytest.raises((ValueError, TypeError)) as e:
                call(logits, out=out)
            assert "out" in str(e.value)
