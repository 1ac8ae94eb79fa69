"""Operator-level host interface: torch tensors in, HIP kernels underneath.

``mm8_one`` / ``mm8_three`` / ``wkv_forward`` mirror the reference's native
operators ``torch.ops.rwkv.*`` (reference
src/rwkvstic/agnostic/backends/cuda/wrapper.cpp:45-127): same names, argument
order and in-place semantics.  ``register_torch_ops()`` publishes them under
the same ``rwkv::`` namespace so reference-style modules resolve them.

Every function requires CUDA (ROCm) tensors and raises on anything else;
nothing here falls back to torch arithmetic.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _native as N

_scratch: dict = {}


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _req(t: torch.Tensor, dtype, name: str) -> None:
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise ValueError(f"{name} must be a CUDA tensor")
    if t.dtype != dtype:
        raise TypeError(f"{name} must be {dtype}, got {t.dtype}")


def _contig(t: torch.Tensor, name: str) -> None:
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


def _workspace(nbytes: int, device) -> torch.Tensor:
    """Scratch of one product, from torch's allocator: it belongs to the stream the call runs on, so that calls of other streams
    have others.  A call that is recorded, or runs on another device than its tensors', takes a buffer kept per device: it may be
    replayed at any time, so where a larger one is needed the smaller ones stay (each at least twice the one before)."""
    here = torch.cuda.current_device()
    key = device.index if device.index is not None else here
    if key == here and not torch.cuda.is_current_stream_capturing():
        return torch.empty(max(nbytes, 1), dtype=torch.uint8, device=device)
    kept = _scratch.setdefault(key, [])
    if not kept or kept[-1].numel() < nbytes:
        kept.append(torch.empty(max(nbytes, 2 * kept[-1].numel() if kept else 1 << 20), dtype=torch.uint8, device=device))
    return kept[-1]


# ---------------------------------------------------------------- reference operators
def _mm8_dtype(x: torch.Tensor, others, what: str) -> torch.dtype:
    """float32 or float64, shared by x, y and r (the dispatch of wrapper.cpp:58-60)."""
    if x.dtype not in (torch.float32, torch.float64):
        raise TypeError(f"{what}: x, y, r must be float32 or float64, got {x.dtype}")
    for t in others:
        _req(t, x.dtype, "x/y/r")
    return x.dtype


def _holds(t: torch.Tensor, n: int) -> bool:
    """Whether the kernels may read or write ``n`` values one after the other from the tensor's first on (a view can have as
    many elements and less memory)."""
    return t.numel() >= n and t.untyped_storage().nbytes() // t.element_size() - t.storage_offset() >= n


def mm8_one(N_in: int, M_out: int, x: torch.Tensor, w: torch.Tensor, y: torch.Tensor, r: torch.Tensor) -> None:
    """``y[k] += sum_j x[j]*(w[j,k]*r[j])``; argument meaning of wrapper.cpp:52-54 (N=in, M=out); x, y, r all
    float32 or all float64 (wrapper.cpp:60-77)."""
    dt = _mm8_dtype(x, (x, y, r), "mm8_one"); _req(w, torch.uint8, "w")
    if x.dim() != 1 or x.stride(0) != 1 or y.stride(0) != 1 or w.dim() != 2 or w.stride(1) != 1:
        raise ValueError("mm8_one: x, y need unit stride and w.stride(1) == 1 (wrapper.cpp:55-57)")
    if not (_holds(x, N_in) and _holds(r, N_in) and _holds(y, M_out)) or w.shape[0] < N_in or w.shape[1] < M_out:
        raise ValueError("mm8_one: tensor smaller than (N, M)")
    L = N.lib()
    f64 = dt == torch.float64
    ws = _workspace((L.rwkv_mm8_f64_workspace_bytes if f64 else L.rwkv_mm8_workspace_bytes)(N_in, M_out, 1), x.device)
    N.check((L.rwkv_mm8_one_f64 if f64 else L.rwkv_mm8_one)(_stream(), N_in, M_out, x.data_ptr(), w.data_ptr(), w.stride(0),
                                                            y.data_ptr(), r.data_ptr(), ws.data_ptr(), ws.numel()))


def mm8_three(N_in: int, M_out: int, x0, x1, x2, w0, w1, w2, y0, y1, y2, r0, r1, r2) -> None:
    """Three ``mm8_one`` problems in one call (wrapper.cpp:82-86); float32 or float64 like ``mm8_one``."""
    dt = _mm8_dtype(x0, (x0, x1, x2, y0, y1, y2, r0, r1, r2), "mm8_three")
    for t in (x0, x1, x2, y0, y1, y2, r0, r1, r2):
        if t.stride(0) != 1:
            raise ValueError("mm8_three: x, y, r need unit stride")
    if not (all(_holds(t, N_in) for t in (x0, x1, x2, r0, r1, r2)) and all(_holds(t, M_out) for t in (y0, y1, y2))):
        raise ValueError("mm8_three: tensor smaller than (N, M)")
    for t in (w0, w1, w2):
        _req(t, torch.uint8, "w")
        if t.dim() != 2 or t.stride(1) != 1 or t.shape[0] < N_in or t.shape[1] < M_out:
            raise ValueError("mm8_three: w must be [>=N, >=M] with unit inner stride")
    L = N.lib()
    f64 = dt == torch.float64
    ws = _workspace((L.rwkv_mm8_f64_workspace_bytes if f64 else L.rwkv_mm8_workspace_bytes)(N_in, M_out, 3), x0.device)
    N.check((L.rwkv_mm8_three_f64 if f64 else L.rwkv_mm8_three)(
        _stream(), N_in, M_out, x0.data_ptr(), x1.data_ptr(), x2.data_ptr(),
        w0.data_ptr(), w0.stride(0), w1.data_ptr(), w1.stride(0), w2.data_ptr(), w2.stride(0),
        y0.data_ptr(), y1.data_ptr(), y2.data_ptr(),
        r0.data_ptr(), r1.data_ptr(), r2.data_ptr(), ws.data_ptr(), ws.numel()))


def wkv_forward(B: int, T: int, C: int, w, u, k, v, y, aa, bb, pp) -> None:
    """float64 WKV with the reference's state convention (wrapper.cpp:45-50)."""
    for name, t in (("w", w), ("u", u), ("k", k), ("v", v), ("y", y), ("aa", aa), ("bb", bb), ("pp", pp)):
        _req(t, torch.float64, name); _contig(t, name)
    if k.numel() < B * T * C or v.numel() < B * T * C or y.numel() < B * T * C:
        raise ValueError("wkv_forward: k/v/y smaller than B*T*C")
    if min(aa.numel(), bb.numel(), pp.numel()) < B * C or min(w.numel(), u.numel()) < C:
        raise ValueError("wkv_forward: state or w/u too small")
    N.check(N.lib().rwkv_wkv_forward_f64(_stream(), B, T, C, w.data_ptr(), u.data_ptr(), k.data_ptr(),
                                         v.data_ptr(), y.data_ptr(), aa.data_ptr(), bb.data_ptr(), pp.data_ptr()))


_registered = False
_SCHEMAS = (
    "wkv_forward(int B, int T, int C, Tensor(a!) w, Tensor(b!) u, Tensor(c!) k, Tensor(d!) v, Tensor(e!) y, Tensor(f!) aa, "
    "Tensor(g!) bb, Tensor(h!) pp) -> ()",
    "mm8_one(int N, int M, Tensor(a!) x, Tensor(b!) w, Tensor(c!) y, Tensor(d!) r) -> ()",
    "mm8_three(int N, int M, Tensor(a!) x, Tensor(b!) x1, Tensor(c!) x2, Tensor(d!) w, Tensor(e!) w1, Tensor(f!) w2, "
    "Tensor(g!) y, Tensor(h!) y1, Tensor(i!) y2, Tensor(j!) r, Tensor(k!) r1, Tensor(l!) r2) -> ()",
)


def register_torch_ops() -> None:
    """Publish ``torch.ops.rwkv.{wkv_forward,mm8_one,mm8_three}`` with the
    reference's schemas (wrapper.cpp:131-141: TORCH_LIBRARY(rwkv, m)).  Their calls run in csrc/rwkv_torch.cpp; what does not
    fit there comes back to the functions above, and all calls do where it is not built."""
    global _registered
    if _registered:
        return
    host = N.host()
    if host is not None:
        host.register_ops(_SCHEMAS)
    else:
        lib = torch.library.Library("rwkv", "DEF")
        for schema in _SCHEMAS:
            lib.define(schema)
        for fn in (wkv_forward, mm8_one, mm8_three):
            lib.impl(fn.__name__, fn, "CUDA")
        register_torch_ops._lib = lib     # keep alive
    _registered = True


# ---------------------------------------------------------------- quantiser / layouts
def _quantize(weight: torch.Tensor, codes: bool, packed: bool, packed16: bool):
    """One quantising pass, its codes written in the layouts asked for (None for the others)."""
    _req(weight, torch.float32, "weight"); _contig(weight, "weight")
    n_out, n_in = weight.shape
    L, dev = N.lib(), weight.device
    c = torch.empty((n_in, n_out), dtype=torch.uint8, device=dev) if codes else None
    p = torch.empty(L.rwkv_packed_bytes(n_in, n_out), dtype=torch.uint8, device=dev) if packed else None
    p16 = torch.empty(L.rwkv_packed_m16_bytes(n_in, n_out), dtype=torch.uint8, device=dev) if packed16 else None
    rng = torch.empty(n_in, dtype=torch.float32, device=dev)
    off = torch.empty(n_in, dtype=torch.float64, device=dev)
    ws = torch.empty(L.rwkv_quantize_workspace_bytes(n_out, n_in), dtype=torch.uint8, device=dev)
    N.check(L.rwkv_quantize_layouts(_stream(), weight.data_ptr(), n_out, n_in, c.data_ptr() if codes else None,
                                    p.data_ptr() if packed else None, p16.data_ptr() if packed16 else None,
                                    rng.data_ptr(), off.data_ptr(), ws.data_ptr(), ws.numel()))
    return c, p, p16, rng, off


def quantize(weight: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """``weight[out, in]`` float32 -> ``(codes[in, out] uint8, range[in] float32, offset[in] float64)``
    (MM8.QuantizeMatrix, matmul.py:24-40)."""
    _req(weight, torch.float32, "weight"); _contig(weight, "weight")
    n_out, n_in = weight.shape
    # One launch without a workspace, with the same bits, where it is no slower than three that cut the matrix both ways.  It
    # walks the rows with a workgroup per 64 channels; us of both, 144 / 192 / 208 / 256 rows: of 64 to 8192 channels 18 / 21 / 25 / 28
    # against 20, of 1 channel 16 / 18 / 21 / 23 against 20; 16384 channels 19 / 22 / 25 / 28 against 22 / 23 / 26 / 27; 65536
    # channels 35 / 43 / 49 / 56 against 62 / 65 / 76 / 80.  (64 rows 12 against 18.5.)
    if n_out > max(200, n_in // 64):
        codes, _, _, rng, off = _quantize(weight, True, False, False)
        return codes, rng, off
    codes = torch.empty((n_in, n_out), dtype=torch.uint8, device=weight.device)
    rng = torch.empty(n_in, dtype=torch.float32, device=weight.device)
    off = torch.empty(n_in, dtype=torch.float64, device=weight.device)
    N.check(N.lib().rwkv_quantize_u8(_stream(), weight.data_ptr(), n_out, n_in, codes.data_ptr(), rng.data_ptr(), off.data_ptr()))
    return codes, rng, off


def quantize_packed(weight: torch.Tensor, m16: bool = True):
    """``quantize`` without the intermediate codes: ``(packed, packed16 or None, range, offset)``, the layouts being
    those of ``pack`` and (``m16``) ``pack_m16``."""
    _, packed, packed16, rng, off = _quantize(weight, False, True, m16)
    return packed, packed16, rng, off


def pack(codes: torch.Tensor) -> torch.Tensor:
    """Reference layout ``codes[in, out]`` -> streaming block layout (1-D uint8)."""
    _req(codes, torch.uint8, "codes")
    if codes.dim() != 2 or codes.stride(1) != 1:
        raise ValueError("codes must be 2-D with unit inner stride")
    n_in, n_out = codes.shape
    L = N.lib()
    packed = torch.empty(L.rwkv_packed_bytes(n_in, n_out), dtype=torch.uint8, device=codes.device)
    N.check(L.rwkv_pack_u8(_stream(), codes.data_ptr(), codes.stride(0), n_in, n_out, packed.data_ptr()))
    return packed


def unpack(packed: torch.Tensor, n_in: int, n_out: int) -> torch.Tensor:
    _req(packed, torch.uint8, "packed"); _contig(packed, "packed")
    L = N.lib()
    if packed.numel() < L.rwkv_packed_bytes(n_in, n_out):
        raise ValueError("packed buffer too small")
    codes = torch.empty((n_in, n_out), dtype=torch.uint8, device=packed.device)
    N.check(L.rwkv_unpack_u8(_stream(), packed.data_ptr(), n_in, n_out, codes.data_ptr(), n_out))
    return codes


def pack_m16(codes: torch.Tensor) -> torch.Tensor:
    """Reference layout ``codes[in, out]`` -> 16x64 signed blocks for the matrix-core decode kernel."""
    _req(codes, torch.uint8, "codes")
    if codes.dim() != 2 or codes.stride(1) != 1:
        raise ValueError("codes must be 2-D with unit inner stride")
    n_in, n_out = codes.shape
    L = N.lib()
    packed = torch.empty(L.rwkv_packed_m16_bytes(n_in, n_out), dtype=torch.uint8, device=codes.device)
    N.check(L.rwkv_pack_m16(_stream(), codes.data_ptr(), codes.stride(0), n_in, n_out, packed.data_ptr()))
    return packed


def unpack_m16(packed: torch.Tensor, n_in: int, n_out: int) -> torch.Tensor:
    _req(packed, torch.uint8, "packed"); _contig(packed, "packed")
    L = N.lib()
    if packed.numel() < L.rwkv_packed_m16_bytes(n_in, n_out):
        raise ValueError("packed buffer too small")
    codes = torch.empty((n_in, n_out), dtype=torch.uint8, device=packed.device)
    N.check(L.rwkv_unpack_m16(_stream(), packed.data_ptr(), n_in, n_out, codes.data_ptr(), n_out))
    return codes


def dequant_packed(packed, rng, off, n_in: int, n_out: int) -> torch.Tensor:
    _req(packed, torch.uint8, "packed"); _req(rng, torch.float32, "range"); _req(off, torch.float64, "offset")
    L = N.lib()
    if packed.numel() < L.rwkv_packed_bytes(n_in, n_out) or rng.numel() < n_in or off.numel() < n_in:
        raise ValueError("buffer too small")
    dq = torch.empty((n_in, n_out), dtype=torch.float32, device=packed.device)
    N.check(L.rwkv_dequant_packed(_stream(), packed.data_ptr(), rng.data_ptr(), off.data_ptr(), n_in, n_out,
                                  dq.data_ptr()))
    return dq


# ---------------------------------------------------------------- stand-alone kernels
def _buffer(t: torch.Tensor, dtype, n: int, name: str) -> None:
    """``n`` values that the kernels read or write one after the other."""
    _req(t, dtype, name); _contig(t, name)
    if t.numel() < n:
        raise ValueError(f"{name} too small")


def _matvec_args(x, packed, packed_bytes: int, n_in: int, n_out: int, r_row, m_row, r_col, m_col, out) -> torch.Tensor:
    """Checks what ``mm8_packed`` and ``mm8_m16`` are given; returns the tensor their results go to."""
    _req(x, torch.float32, "x"); _contig(x, "x")
    if x.dim() != 2 or x.shape[1] != n_in:
        raise ValueError("x must be [B, n_in]")
    _buffer(packed, torch.uint8, packed_bytes, "packed weights")
    _buffer(r_row, torch.float32, n_in, "r_row"); _buffer(m_row, torch.float64, n_in, "m_row")
    for t, nm in ((r_col, "r_col"), (m_col, "m_col")):
        if t is not None:
            _buffer(t, torch.float32, n_out, nm)
    y = out if out is not None else torch.empty((x.shape[0], n_out), dtype=torch.float64, device=x.device)
    _buffer(y, torch.float64, x.shape[0] * n_out, "out")
    return y


def mm8_packed(x: torch.Tensor, packed: torch.Tensor, n_in: int, n_out: int,
               r_row: torch.Tensor, m_row: torch.Tensor,
               r_col: Optional[torch.Tensor] = None, m_col: Optional[torch.Tensor] = None,
               out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``y[B, out]`` float64 for ``x[B, in]`` float32, B in {1, 2, 4, 8}."""
    host = N.host()
    y = host and host.mm8_packed(x, packed, n_in, n_out, r_row, m_row, r_col, m_col, out)
    if y is not None:
        return y
    L = N.lib()
    y = _matvec_args(x, packed, L.rwkv_packed_bytes(n_in, n_out), n_in, n_out, r_row, m_row, r_col, m_col, out)
    B = x.shape[0]
    N.check(L.rwkv_mm8_packed(_stream(), B, n_in, n_out, x.data_ptr(), packed.data_ptr(), r_row.data_ptr(),
                              m_row.data_ptr(), r_col.data_ptr() if r_col is not None else None,
                              m_col.data_ptr() if m_col is not None else None, y.data_ptr()))
    return y


def mm8_m16(x: torch.Tensor, packed16: torch.Tensor, n_in: int, n_out: int,
            r_row: torch.Tensor, m_row: torch.Tensor,
            r_col: Optional[torch.Tensor] = None, m_col: Optional[torch.Tensor] = None,
            out: Optional[torch.Tensor] = None, workspace: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``mm8_packed`` on the matrix cores: ``y[B, out]`` float64 for ``x[B, in]`` float32, any B in 1..8, weights in
    the M16 layout (``pack_m16``); exact integer sums instead of float32 accumulation."""
    host = N.host()
    y = host and host.mm8_m16(x, packed16, n_in, n_out, r_row, m_row, r_col, m_col, out, workspace)
    if y is not None:
        return y
    L = N.lib()
    y = _matvec_args(x, packed16, L.rwkv_packed_m16_bytes(n_in, n_out), n_in, n_out, r_row, m_row, r_col, m_col, out)
    B = x.shape[0]
    need = L.rwkv_mm8_m16_workspace_bytes(B, n_in)
    ws = workspace if workspace is not None else torch.empty(max(need, 1), dtype=torch.uint8, device=x.device)
    _buffer(ws, ws.dtype, 0, "workspace")               # (its bytes are counted by the library)
    N.check(L.rwkv_mm8_m16(_stream(), B, n_in, n_out, x.data_ptr(), packed16.data_ptr(), r_row.data_ptr(),
                           m_row.data_ptr(), r_col.data_ptr() if r_col is not None else None,
                           m_col.data_ptr() if m_col is not None else None, y.data_ptr(), ws.data_ptr(), ws.numel()))
    return y


def gemm8(x: torch.Tensor, packed16: torch.Tensor, rng: torch.Tensor, off: torch.Tensor,
          n_in: int, n_out: int) -> torch.Tensor:
    """``y[T, n_out] = x[T, n_in] @ dequantised matrix`` with the single-token arithmetic
    (fp32(x*range) as exact fixed point, integer dot products, float64 zero-point term);
    the T > 1 branch of MM8.forward (matmul.py:56-57) without its bfloat16 rounding."""
    _req(x, torch.float64, "x"); _contig(x, "x")
    _req(packed16, torch.uint8, "packed16"); _req(rng, torch.float32, "range"); _req(off, torch.float64, "offset")
    if x.dim() != 2 or x.shape[1] != n_in:
        raise ValueError("gemm8: x must be [T, n_in]")
    T = x.shape[0]
    L = N.lib()
    if packed16.numel() < L.rwkv_packed_m16_bytes(n_in, n_out) or rng.numel() < n_in or off.numel() < n_in:
        raise ValueError("gemm8: matrix buffers smaller than (n_in, n_out)")
    y = torch.empty((T, n_out), dtype=torch.float64, device=x.device)
    ws = _workspace(L.rwkv_gemm8_workspace_bytes(T, n_in, n_out), x.device)
    N.check(L.rwkv_gemm8(_stream(), T, n_in, n_out, x.data_ptr(), packed16.data_ptr(), rng.data_ptr(),
                         off.data_ptr(), y.data_ptr(), ws.data_ptr(), ws.numel()))
    return y


def wkv_f32(w, u, k, v, aa, bb, pp) -> torch.Tensor:
    """Max-shifted float32 WKV; ``k, v`` are ``[B, T, C]``; state ``[B, C]`` updated in place."""
    host = N.host()
    y = host and host.wkv_f32(w, u, k, v, aa, bb, pp)
    if y is not None:
        return y
    for name, t in (("w", w), ("u", u), ("k", k), ("v", v), ("aa", aa), ("bb", bb), ("pp", pp)):
        _req(t, torch.float32, name); _contig(t, name)
    if k.dim() != 3 or v.shape != k.shape:
        raise ValueError("k, v must be [B, T, C]")
    B, T, Cn = k.shape
    if min(aa.numel(), bb.numel(), pp.numel()) < B * Cn or min(w.numel(), u.numel()) < Cn:
        raise ValueError("state or w/u too small")
    y = torch.empty_like(k)
    N.check(N.lib().rwkv_wkv_f32(_stream(), B, T, Cn, w.data_ptr(), u.data_ptr(), k.data_ptr(), v.data_ptr(),
                                 y.data_ptr(), aa.data_ptr(), bb.data_ptr(), pp.data_ptr()))
    return y


def sample_token(logits: torch.Tensor, *, greedy: bool = False, temp: float = 1.0, tau: float = 0.8, end_adj: float = 0.0,
                 seed: int = 0, counter: int = 0, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """One choice of the device-side sampler (typical.py:1-17; ``logits[0] += end_adj`` in place first,
    rwkvMaster.py:37); the uniform number is a hash of ``(seed, counter)``."""
    _req(logits, torch.float64, "logits"); _contig(logits, "logits")
    out = out if out is not None else torch.empty(1, dtype=torch.int64, device=logits.device)
    _buffer(out, torch.int64, 1, "out")
    N.check(N.lib().rwkv_sample_token(_stream(), logits.data_ptr(), logits.numel(), 1 if greedy else 0, float(temp),
                                      float(tau), float(end_adj), int(seed) & (2 ** 64 - 1), int(counter), out.data_ptr()))
    return out


def argmax(logits: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    _req(logits, torch.float64, "logits"); _contig(logits, "logits")
    out = out if out is not None else torch.empty(1, dtype=torch.int64, device=logits.device)
    _buffer(out, torch.int64, 1, "out")
    N.check(N.lib().rwkv_argmax_f64(_stream(), logits.data_ptr(), logits.numel(), out.data_ptr()))
    return out
