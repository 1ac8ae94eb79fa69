"""Slices of a product added up by the LayerNorm kernel against the same product finished before it: the residual, the shift rows and the
quantised rows that leave that kernel have the same bits.  The library's internal functions by their linkage names."""
import ctypes as C

import pytest
import torch

import product_plans
from rwkvstic_amd import _native

pytestmark = pytest.mark.gpu

P, i64 = C.c_void_p, C.c_int64
ROW_ADD, ROW_GATE_ADD = 2, 3


class Operand(C.Structure):
    _fields_ = [("dig", P), ("S", P), ("qs", P), ("zp", P)]


class Product(C.Structure):
    _fields_ = [("a", Operand), ("w16", P), ("out", P), ("stream", C.c_bool)]


class Deferred(C.Structure):
    _fields_ = [("tot", P), ("slice", C.c_size_t), ("slices", C.c_int), ("ldd", C.c_int), ("op", C.c_int), ("apart", C.c_bool), ("fused", C.c_bool),
                ("S", P), ("qs", P), ("zp", P), ("gate", P)]


class Few(C.Structure):
    _fields_ = [("add", Deferred), ("x_out", P), ("shift_out", P), ("commit_src", P), ("commit_dst", P)]


def _fn(name, *args):
    fn = getattr(_native.lib(), name)
    fn.restype, fn.argtypes = C.c_int, list(args)
    return lambda *a: _native.check(fn(*a))


# (5120 channels: the att output only.  A gated update of theirs rounds the product for itself where slices are handed on.)
@pytest.mark.parametrize("sequence,R,width,K,op", [
    (True, 40, 512, 2048, ROW_GATE_ADD), (True, 127, 1024, 1024, ROW_ADD), (True, 33, 1024, 1024, ROW_ADD), (True, 28, 1024, 4096, ROW_GATE_ADD),
    (True, 80, 1536, 6144, ROW_GATE_ADD), (True, 20, 2048, 8192, ROW_GATE_ADD), (True, 64, 2048, 2048, ROW_ADD),
    (False, 8, 1024, 4096, ROW_GATE_ADD), (False, 7, 1536, 6144, ROW_GATE_ADD), (False, 8, 2560, 10240, ROW_GATE_ADD), (False, 32, 1024, 4096, ROW_GATE_ADD),
    (False, 17, 2560, 10240, ROW_GATE_ADD), (False, 32, 3584, 14336, ROW_GATE_ADD), (False, 32, 5120, 5120, ROW_ADD), (False, 100, 2560, 2560, ROW_ADD),
    (True, 100, 1088, 1088, ROW_ADD), (False, 86, 1536, 1536, ROW_ADD), (False, 127, 2048, 2048, ROW_ADD)])   # (more workgroups than compute units)
def test_slices_handed_on_have_the_bits_of_a_finished_product(sequence, R, width, K, op):
    from rwkvstic_amd import ops
    print(f"handed on: sequence={sequence} R={R} C={width} K={K} op={op}", flush=True)
    assert 1 < product_plans.handed_on(R, width, K, sequence) <= product_plans.DEFER_SLICES
    quant = _fn("_ZN4rwkv10rows_quantEP12ihipStream_tllPKvbPKfPKdRKNS_11RowsOperandEPd", P, i64, i64, P, C.c_bool, P, P, P, P)
    products = _fn("_ZN4rwkv13rows_productsEP12ihipStream_tiPKNS_11RowsProductEPxllliPKfPNS_12RowsDeferredEb",
                   P, C.c_int, P, P, i64, i64, i64, C.c_int, P, P, C.c_bool)
    layernorm = _fn("_ZN4rwkv17rows_ln_mix_quantEP12ihipStream_tilibPKdS3_S3_S3_S3_PdlPKPKfPKS3_PKNS_11RowsOperandEPKNS_7RowsFewE",
                    P, C.c_int, i64, C.c_int, C.c_bool, P, P, P, P, P, P, i64, P, P, P, P)
    g = torch.Generator(device="cuda").manual_seed(R * 7 + width)
    f64 = dict(generator=g, device="cuda", dtype=torch.float64)
    w16 = ops.pack_m16(torch.randint(0, 256, (K, width), generator=g, dtype=torch.uint8, device="cuda"))
    act, gate = torch.rand(R, K, generator=g, device="cuda"), torch.randn(R, width, generator=g, device="cuda")
    k_range, k_offset = torch.rand(K, generator=g, device="cuda") * 1e-3, torch.randn(K, **f64) * 1e-2
    x, mu = torch.randn(R, width, **f64), torch.rand(3, width, **f64)
    ln_w, ln_b, prev = torch.rand(width, **f64) + 0.5, torch.randn(width, **f64), torch.randn(R, width, **f64)
    ranges, offsets = torch.rand(3, width, generator=g, device="cuda") * 1e-3, torch.randn(3, width, **f64) * 1e-2
    st = torch.cuda.current_stream().cuda_stream
    keep = []

    def buffer(n):                                          # (zeroed: digits of rows past the last one are multiplied too)
        keep.append(torch.zeros(n, dtype=torch.uint8, device="cuda"))
        return keep[-1]

    def operand(k):
        parts = [buffer(-(-R // 4) * (k // 64) * 1024)] + [buffer(R * 8) for _ in range(3)]
        return parts, Operand(*[p.data_ptr() for p in parts])

    _, a = operand(K)
    tot = buffer(product_plans.pass_tot_bytes(R, width, K, 16, 1))      # (the quantiser's scratch as well)
    quant(st, R, K, act.data_ptr(), True, k_range.data_ptr(), k_offset.data_ptr(), C.byref(a), tot.data_ptr())

    def one_way(handed):
        # finished: x is updated in place; handed on: it stays, and the LayerNorm kernel leaves the new one in another buffer
        xin, xout, shift = x.clone(), torch.zeros_like(x), torch.zeros_like(x)
        few = Few()
        p = Product(a, w16.data_ptr(), xin.data_ptr(), False)
        products(st, 1, C.byref(p), tot.data_ptr(), R, K, width, op, gate.data_ptr(), C.byref(few.add) if handed else None, sequence)
        assert (few.add.tot is not None) == handed
        few.x_out, few.shift_out = xout.data_ptr() if handed else None, shift.data_ptr()
        outs = [operand(width) for _ in range(3)]
        table = lambda t: C.byref((P * 3)(*[t[m].data_ptr() for m in range(3)]))
        layernorm(st, 3, R, width, sequence, xin.data_ptr(), ln_w.data_ptr(), ln_b.data_ptr(), mu.data_ptr(), prev.data_ptr(), shift.data_ptr(), width,
                  table(ranges), table(offsets), C.byref((Operand * 3)(*[o for _, o in outs])), C.byref(few))
        torch.cuda.synchronize()
        assert torch.equal(xin, x) == handed
        return [xout if handed else xin, shift] + [b for parts, _ in outs for b in parts]

    for i, (want, got) in enumerate(zip(one_way(False), one_way(True))):
        assert torch.equal(want, got), i
    assert not torch.equal(want, torch.zeros_like(want))
