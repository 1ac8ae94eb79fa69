"""Host-only checks of the workspace sizing of the many-row products: whatever kernel variant and number of
contraction splits the launch plan picks, the integer totals it writes (one slice per split and product) fit
the buffer the sizing functions reserve.  Nothing is launched; no GPU needed."""
import ctypes as C
import os

import pytest

import product_plans


@pytest.fixture(scope="module")
def lib():
    import shutil
    from rwkvstic_amd import _native
    if not os.path.exists(_native.LIB_PATH):
        if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
            pytest.skip("librwkv_hip.so is not built and there is no hipcc to build it with")
        from rwkvstic_amd import build
        build.build(verbose=False)
    return _native.lib()


def _plan(lib, T, K, N, n):
    plan = (C.c_int * 4)()
    tot = C.c_size_t()
    assert lib.rwkv_gemm8_plan(T, K, N, n, C.byref(plan), C.byref(tot)) == 0, lib.rwkv_last_error()
    return tuple(plan), tot.value


ROWS = list(range(1, 40)) + [47, 48, 63, 64, 65, 100, 127, 128, 129, 255, 256, 257, 300, 400, 511, 512, 513, 640,
                             700, 768, 769, 800, 832, 896, 960, 961, 1000, 1023, 1024]
WIDTHS = [16, 64, 72, 256, 512, 768, 1024, 2048, 2560, 3072, 4096, 5120, 10240, 20480, 50277]
DEPTHS = [64, 512, 1024, 2560, 5120, 10240, 20480]


def test_totals_buffer_holds_every_slice(lib):
    worst = 0
    for T in ROWS:
        for N in WIDTHS:
            slice_bytes = -(-T // 4) * 4 * (-(-N // 16) * 16) * 8
            for K in DEPTHS:
                for n in (1, 2, 3):
                    (kind, gx, gy, split), tot = _plan(lib, T, K, N, n)
                    assert 1 <= split <= 8 and kind in (0, 1, 2, 3)
                    assert split * slice_bytes <= tot, (T, K, N, n, kind, split, tot)
                    worst = max(worst, split)
    assert worst > 1          # the sweep does reach split contractions


def test_split_contractions_are_where_the_grid_is_small(lib):
    """A split contraction costs a second launch, so only grids far below the device split: [800 x 2560] x
    [2560 x 2560] takes the 64 x 160 variant (208 workgroups) unsplit with the tail in its epilogue, the same
    product for 250 rows (80 workgroups of 64 x 128) splits in two, for 60 rows (20 workgroups) in four (parts of
    at least 8 contraction blocks)."""
    (kind, gx, gy, split), tot = _plan(lib, 800, 2560, 2560, 1)
    assert kind == 3 and split == 1 and gx * gy == 208
    (kind, gx, gy, split), tot = _plan(lib, 250, 2560, 2560, 1)
    assert kind == 2 and split == 2 and gx * gy == 80
    assert split * 252 * 2560 * 8 <= tot
    (kind, gx, gy, split), tot = _plan(lib, 60, 2560, 2560, 1)
    assert kind == 2 and split == 4 and split * 60 * 2560 * 8 <= tot
    # a contraction of 200 blocks and more splits once while the grid is below the device: the ffn value product of
    # the 14B shape on a 256-token chunk (160 workgroups), not the same width's [5120 x 5120] products
    (kind, gx, gy, split), tot = _plan(lib, 256, 20480, 5120, 1)
    assert kind == 2 and gx * gy == 160 and split == 2 and split * 256 * 5120 * 8 <= tot
    assert _plan(lib, 256, 5120, 5120, 1)[0][3] == 1


@pytest.mark.parametrize("T", [1, 4, 5, 8])
def test_few_rows_reserve_the_slices_they_write(lib, T):
    """At most 8 rows run whole contractions up to 65536, so the totals of one slice are reserved, and those of the slices
    there are beyond: for a head of 50277 columns eight slices are 13 MB of workspace in every forward call."""
    for K, N, n in ((5120, 50277, 1), (20480, 5120, 1), (2560, 2560, 3), (65536, 16, 1), (65537 + 63, 16, 1), (4 * 65536, 300, 1)):
        slice_bytes = -(-T // 4) * 4 * (-(-N // 16) * 16) * 8
        (kind, gx, gy, split), tot = _plan(lib, T, K, N, n)
        assert kind == 0 and split == (1 if K <= 65536 else 2 if K <= 2 * 65536 else 4) and tot == split * slice_bytes, (K, N)


def test_gemm8_workspace_covers_quantiser_scratch(lib):
    """A few rows of a long contraction are quantised in parts whose records sit in the totals area."""
    for T in (1, 4, 8):
        for K in (8192, 20480, 131072, 1 << 20):
            need = T * -(-K // (4 * 256 * 3)) * 16
            fixed = 3 * (-(-T * 8 // 256) * 256) + (-(-(-(-T // 4) * (K // 64) * 1024) // 256) * 256)
            assert lib.rwkv_gemm8_workspace_bytes(T, K, 16) - fixed >= need, (T, K)


@pytest.mark.parametrize("C_,F", [(64, 64), (512, 2048), (768, 640), (1024, 4096), (1024, 8192), (1024, 16384), (1536, 20480), (2048, 512), (2560, 10240),
                                  (4096, 16384), (5120, 640), (5120, 20480)])
def test_totals_of_a_pass_hold_those_of_every_product_in_it(lib, C_, F):
    """Whatever the order of n_embd, n_ffn and the vocabulary: fewer columns may be cut in slices where more are not.  Of a prompt longer
    than a pass the last one may have any number of rows."""
    def need(rows, K, N, n):
        (kind, gx, gy, split), _ = _plan(lib, rows, K, N, n)
        return n * split * (-(-rows // 4) * 4 * (-(-N // 16) * 16) * 8)

    layers = {R: max(need(R, C_, C_, 3), need(R, C_, F, 1), need(R, F, C_, 1)) for R in ROWS}
    for V in (16, 100, 1000, 4000, 8000, 14000, 16000, 20000, 50277, 65536):
        one = need(1, C_, V, 1)
        for R in ROWS:
            assert max(layers[R], need(R, C_, V, 1)) <= product_plans.pass_tot_bytes(R, C_, F, V, R), (V, R)
            assert max(layers[R], one) <= product_plans.pass_tot_bytes(R, C_, F, V, 1), (V, R)
        assert max(layers.values()) <= product_plans.pass_tot_bytes(1024, C_, F, V, 1), V


@pytest.mark.parametrize("C_", [64, 320, 512, 768, 1024, 1088, 1536, 2048, 2112, 2560, 3072, 3584, 4096, 5120, 6144])
def test_slices_left_to_the_next_kernel_are_whole_and_fit(lib, C_):
    """The plans of k, v, r and of the two residual updates, which depend on who adds up the slices: the totals hold all of them, no slice is
    empty (nothing would be written for it), and a few-row product has its kernel."""
    most = 0
    for F in (64, 640, 2 * C_, 4 * C_, 16384):
        for R in ROWS:
            for sequence in (False, True):
                room, who = product_plans.pass_tot_bytes(R, C_, F, 16, 1 if sequence else R), product_plans.readers(R, C_, sequence)
                for K, n, readers in ((C_, 1, who), (F, 1, who), (C_, 3, int(who == 1))):
                    kind, _, _, s = product_plans.plan(R, K, C_, n, readers)
                    MT, NT, KB = -(-R // 4), -(-C_ // 16), K // 64
                    each = -(-KB // s)
                    assert n * s * MT * 4 * NT * 16 * 8 <= room, (F, R, K, n, s)
                    assert (s - 1) * each < KB, (F, R, K, n, s)
                    if kind == product_plans.VEC:
                        assert product_plans.vec_kernel(MT, NT * s * n, KB, each), (F, R, K, n, s)
                    if readers:
                        most = max(most, s)
    assert most > 1 or C_ <= 320


def test_slices_of_9_to_32_rows_fit_each_xcd(lib):
    """More slices must leave the compute units of the XCD that has the most column blocks (of eight tiles, dealt out in turn) less to draw:
    rounds of 32 workgroups, times the blocks of one."""
    seen = set()
    for C_ in range(256, 6145, 64):
        for R in (9, 16, 17, 32):
            for K, n, readers in ((C_, 3, 1), (C_, 1, 1), (4 * C_, 1, 1), (C_, 1, 0), (C_, 1, 2), (4 * C_, 1, 2)):
                kind, gx, _, s = product_plans.plan(R, K, C_, n, readers)
                if kind == product_plans.SKINNY and s > 1:
                    assert gx == -(-C_ // 128)
                    draw = [-(-(-(-gx // 8) * n * t) // 32) * -(-(K // 64) // t) for t in range(1, s + 1)]
                    assert draw[-1] == min(draw), (C_, R, K, n, s, draw)
                    seen.add(s)
    assert {2, 3, 4, 5, 6} <= seen


def test_what_is_handed_on(lib):
    """Short prompts of narrow models and batches of fewer than 128 rows; slices by what they save, no more than the next kernel takes."""
    assert [product_plans.readers(R, C_, s) for R, C_, s in ((127, 5120, False), (128, 512, False), (127, 1024, True), (128, 512, True), (64, 2048, True),
                                                             (65, 2048, True), (4, 2112, True))] == [1, 0, 2, 0, 2, 0, 0]
    assert [product_plans.handed_on(R, 2560, 10240) for R in (4, 8, 16, 17, 32, 127)] == [0, 3, 0, 6, 6, 4]
    assert [product_plans.handed_on(77, C_, K, True) for C_, K in ((512, 512), (512, 2048), (1024, 1024), (1024, 4096), (1536, 6144))] == [0, 4, 2, 0, 4]


def test_a_pending_product_keeps_its_row_constants_apart(lib):
    """Few rows: a row of the LayerNorm kernel has one workgroup per mix, all of which read S, qs and zp of a product handed on
    unfinished; outputs in the same arrays would be written by one while another still reads.  The call is refused on the
    host, before anything is launched, for each of the three arrays and each output."""
    P, i64, D = C.c_void_p, C.c_int64, C.c_void_p

    class Operand(C.Structure):
        _fields_ = [("dig", P), ("S", P), ("qs", P), ("zp", P)]

    class Deferred(C.Structure):
        _fields_ = [("tot", P), ("slice", C.c_size_t), ("slices", C.c_int), ("ldd", C.c_int), ("op", C.c_int),
                    ("S", P), ("qs", P), ("zp", P), ("gate", P)]

    class Few(C.Structure):
        _fields_ = [("add", Deferred), ("x_out", P), ("shift_out", P), ("commit_src", P), ("commit_dst", P)]

    fn = getattr(lib, "_ZN4rwkv17rows_ln_mix_quantEP12ihipStream_tilibPKdS3_S3_S3_S3_PdlPKPKfPKS3_PKNS_11RowsOperandEPKNS_7RowsFewE")
    fn.restype, fn.argtypes = C.c_int, [P, C.c_int, i64, C.c_int, C.c_bool, D, D, D, D, D, D, i64, P, P, P, P]
    ptrs = (P * 3)(16, 16, 16)
    for n_mix in (2, 3):
        for k in range(n_mix):
            for field in ("S", "qs", "zp"):
                out = (Operand * 3)(*[Operand(16, 1024 * (i + 1), 1024 * (i + 1) + 256, 1024 * (i + 1) + 512) for i in range(3)])
                few = Few(Deferred(16, 0, 1, 64, 2, 8192, 8448, 8704, None), 32, 48, None, None)     # op 2: ROW_ADD
                setattr(few.add, field, getattr(out[k], field))
                assert fn(None, n_mix, 100, 64, False, 64, 16, 16, 16, 16, 16, 320, ptrs, ptrs, C.byref(out), C.byref(few)) == -1
                assert b"row constants" in lib.rwkv_last_error(), (n_mix, k, field)


def test_every_few_row_product_has_its_kernel_and_every_kernel_a_product(lib):
    """gemv16_kernel: the rules that say which products it takes and in which shape, against the list of its instances."""
    import re
    plan, tot = (C.c_int * 4)(), C.c_size_t()
    reached = set()
    for MT in range(1, 9):
        for tiles in list(range(1, 60)) + [100, 127, 128, 200, 255, 256, 257, 300, 319, 320, 321, 400, 511, 512, 513, 900, 1279, 1280, 1281, 2000, 3143, 5000]:
            for KB in list(range(1, 130)) + [160, 175, 176, 200, 233, 234, 240, 320, 350, 351, 512, 700, 701, 1023, 1024, 1025, 2048, 2049]:
                assert lib.rwkv_gemm8_plan(4 * MT, 64 * KB, 16 * tiles, 1, C.byref(plan), C.byref(tot)) == 0
                kind, _, _, split = plan
                at = product_plans.vec_kernel(MT, tiles * split, KB, -(-KB // split))
                assert (kind == 0) == bool(at), (MT, tiles, KB)
                reached.add(at)
    source = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rwkvstic_amd", "csrc", "rwkv_rows.hip")).read()
    assert len(reached - {None}) == 2 * len(re.findall(r"RWKV_VEC(?:12|34|68)\(\d", source))


@pytest.mark.parametrize("C_,layers,vocab", [(512, 208, 65536), (768, 201, 98304), (1024, 200, 65536), (1536, 177, 98304), (2048, 174, 131072),
                                             (2560, 161, 163840), (4096, 123, 262144), (5120, 1000, 163840)])
def test_models_the_token_kernel_takes(lib, C_, layers, vocab):
    """At least so many layers (their state rows lie in LDS), and vocabularies up to a line that stays: a model on the other
    side of it would change kernels, and with them the last bits of its logits."""
    takes = getattr(lib, "_ZN4rwkv16decode_supportedEllll")
    takes.restype, takes.argtypes = C.c_bool, [C.c_int64] * 4
    assert takes(layers, C_, 4 * C_, vocab) and not takes(2, C_, 4 * C_, vocab + 1) and not takes(2, C_, 4 * C_ + 64, vocab)
