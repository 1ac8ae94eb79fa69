"""Host-side view of the plans that the many-row products of a model follow (library internals by their linkage names; nothing is launched)."""
import ctypes as C

from rwkvstic_amd import _native

VEC, SKINNY, GENERAL, WIDE = range(4)       # few rows | 9 to 32 rows | 64 x 128 | 64 x 160 or 64 x 80 columns to a workgroup
DEFER_SLICES = 6                            # more slices than these are added up by a launch of their own


def _fn(name, res, *args):
    fn = getattr(_native.lib(), name)
    fn.restype, fn.argtypes = res, list(args)
    return fn


def readers(rows, C_, sequence):
    """Who adds up the slices of a residual update: 0 a launch of their own, 1 the next kernel, 2 that twice."""
    return _fn("_ZN4rwkv12rows_readersEllb", C.c_int, C.c_int64, C.c_int64, C.c_bool)(rows, C_, sequence)


def plan(rows, K, N, n=1, readers=0):
    """(kernel, grid x, grid y, slices)"""
    out = (C.c_int * 4)()
    _fn("_ZN4rwkv18rows_plan_describeEllliiPi", None, C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_void_p)(rows, K, N, n, readers, C.byref(out))
    return tuple(out)


def handed_on(rows, C_, K, sequence=False):
    """Slices of a residual update of K values a row that the next kernel adds up (0: none, the product or a launch of its own finishes it)."""
    r = readers(rows, C_, sequence)
    slices = plan(rows, K, C_, 1, r)[3]
    return slices if r and 1 < slices <= DEFER_SLICES else 0


def pass_tot_bytes(rows, C_, F, V, head_rows):
    """Bytes of integer totals in the workspace of a pass."""
    return _fn("_ZN4rwkv19rows_pass_tot_bytesElllll", C.c_size_t, *[C.c_int64] * 5)(rows, C_, F, V, head_rows)


def vec_kernel(MT, tiles, KB, kb_per_split):
    """Address of the few-row kernel of a launch (None: there is none)."""
    return _fn("_ZN4rwkv13vec_kernel_ofEllll", C.c_void_p, *[C.c_int64] * 4)(MT, tiles, KB, kb_per_split)
