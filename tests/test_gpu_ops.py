"""GPU parity of the stand-alone operators against the CPU oracle.
Every case goes through the C ABI (rwkvstic_amd.ops -> ctypes -> librwkv_hip.so)."""
import pytest
import torch

from oracle import rwkv_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from rwkvstic_amd import ops as _ops
    return _ops


def _say(msg):
    print(msg, flush=True)


# ------------------------------------------------------------------ quantiser + layouts
@pytest.mark.parametrize("shape", [(8, 8), (5, 3), (300, 130), (3072, 768), (2560, 2560), (1000, 257)])
def test_quantiser_bit_exact_codes_and_1ulp_dequant(ops, shape):
    _say(f"quantise {shape}")
    g = torch.Generator().manual_seed(shape[0] * 7 + shape[1])
    W = torch.randn(*shape, generator=g) * 0.02
    c_ref, r_ref, o_ref = O.quantize_matrix(W)
    codes, rng, off = ops.quantize(W.cuda())
    torch.cuda.synchronize()
    assert torch.equal(codes.cpu(), c_ref), "codes differ"
    assert torch.equal(rng.cpu(), r_ref), "range differs"
    # offset differs only by the summation order of the mean fraction
    assert torch.allclose(off.cpu(), o_ref, rtol=1e-13, atol=1e-300)
    packed = ops.pack(codes)
    assert torch.equal(ops.unpack(packed, *codes.shape).cpu(), c_ref), "pack/unpack round trip"
    dq = ops.dequant_packed(packed, rng, off, *codes.shape).cpu()
    want = O.dequant_canonical(c_ref, r_ref, o_ref)
    ulp = torch.abs(torch.nextafter(want, torch.full_like(want, float("inf"))) - want)
    assert ((dq - want).abs() <= ulp).all(), "dequantised weights differ by more than 1 ulp"


def test_quantiser_constant_channel(ops):
    W = torch.randn(40, 16) * 0.02
    W[:, 3] = 0.125
    codes, rng, off = ops.quantize(W.cuda())
    assert int(codes[3].max()) == 0 and float(rng[3]) == 0.0 and float(off[3]) == 0.125


# one tile, its edges on both sides, several tiles per workgroup, ragged rows that rule out 16-byte loads
@pytest.mark.parametrize("shape", [(1, 1), (64, 128), (63, 127), (65, 129), (300, 132), (1000, 257), (10240, 2560), (50277, 768)])
def test_quantised_layouts_are_the_packed_codes(ops, shape):
    _say(f"quantise to layouts {shape}")
    g = torch.Generator().manual_seed(shape[0] + 5 * shape[1])
    W = (torch.randn(*shape, generator=g) * 0.02).cuda()
    W[:, -1] = 0.25
    codes, rng, off = ops.quantize(W)
    packed, packed16, rng2, off2 = ops.quantize_packed(W)
    assert torch.equal(packed, ops.pack(codes)) and torch.equal(packed16, ops.pack_m16(codes))
    assert torch.equal(rng, rng2) and torch.equal(off, off2)
    assert ops.quantize_packed(W, m16=False)[1] is None
    c_ref, r_ref, o_ref = O.quantize_matrix(W.cpu())
    live = r_ref > 0                                    # (the oracle divides by the range of a constant channel)
    assert torch.equal(codes.cpu()[live], c_ref[live]) and torch.equal(rng.cpu()[live], r_ref[live])
    assert torch.allclose(off.cpu()[live], o_ref[live], rtol=1e-13, atol=1e-300)
    assert int(codes[-1].max()) == 0 and float(off[-1]) == 0.25


# rows on both sides of a tile of the serial sums (96), of the four tiles requested together (384) and of an encoding
# tile (64); channels on both sides of a workgroup's 8 and 128; the rows up to which ops.quantize takes the one and the other; more rows than 65535 encoding tiles of 256
@pytest.mark.parametrize("shape", [(1, 1), (15, 16), (17, 15), (64, 17), (96, 8), (97, 9), (127, 128), (129, 129), (384, 7), (385, 8), (200, 70), (201, 70), (300, 132), (1000, 257),
                                   (2560, 640), (50277, 64), (65535 * 256 + 5, 1)])
def test_both_quantisers_give_the_same_bits(ops, shape):
    """rwkv_quantize_u8 (no workspace, one workgroup per 64 channels) and rwkv_quantize_layouts: codes, ranges and offsets."""
    from rwkvstic_amd import _native as N
    _say(f"quantise twice {shape}")
    n_out, n_in = shape
    g = torch.Generator(device="cuda").manual_seed(n_out + 3 * n_in)
    W = torch.randn(n_out, n_in, generator=g, device="cuda") * 0.02
    if n_in > 2:
        W[:, 1] = 0.25                                  # a constant channel
    codes, _, _, rng, off = ops._quantize(W, True, False, False)
    c = torch.empty_like(codes)
    r, o = torch.empty_like(rng), torch.empty_like(off)
    N.check(N.lib().rwkv_quantize_u8(torch.cuda.current_stream().cuda_stream, W.data_ptr(), n_out, n_in, c.data_ptr(), r.data_ptr(), o.data_ptr()))
    assert torch.equal(codes, c) and torch.equal(rng, r) and torch.equal(off, o)
    assert all(torch.equal(a, b) for a, b in zip(ops.quantize(W), (codes, rng, off)))


def test_layouts_of_more_channels_than_one_launch_has_workgroups_for(ops):
    """Eight channels to a workgroup would be more than the 2^32 threads of a launch; the plain codes of three rows come from
    the one-launch kernel and have the same bits."""
    n_out, n_in = 3, (1 << 27) + 1000
    _say(f"quantise {n_out} x {n_in}")
    g = torch.Generator(device="cuda").manual_seed(5)
    W = torch.randn(n_out, n_in, generator=g, device="cuda") * 0.02
    codes, rng, off = ops.quantize(W)
    packed, packed16, r, o = ops.quantize_packed(W)
    assert torch.equal(rng, r) and torch.equal(off, o)
    assert torch.equal(ops.unpack(packed, n_in, n_out), codes) and torch.equal(ops.unpack_m16(packed16, n_in, n_out), codes)


def test_pack_strided_and_ragged(ops):
    big = torch.randint(0, 256, (200, 400), dtype=torch.uint8, device="cuda")
    view = big[:130, :77]                      # stride 400, ragged in both dims
    packed = ops.pack(view)
    assert torch.equal(ops.unpack(packed, 130, 77), view)


# ------------------------------------------------------------------ packed matvec (isolated workload)
SHAPES = [(2560, 2560), (2560, 10240), (10240, 2560)]


PACKED_CASES = [(n_in, n_out, B) for (n_in, n_out) in SHAPES + [(96, 40), (130, 77), (768, 50277)] for B in (1, 8)]
PACKED_CASES += [(256, 8200, 4), (256, 8200, 2)]     # 1025 column tiles: four per workgroup at B = 4 (ragged last group), one at B = 2


@pytest.mark.parametrize("n_in,n_out,B", PACKED_CASES)
def test_mm8_packed_general_form(ops, n_in, n_out, B):
    _say(f"mm8_packed in={n_in} out={n_out} B={B}")
    g = torch.Generator().manual_seed(n_in + 3 * n_out + B)
    codes = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8)
    m_row = torch.randn(n_in, generator=g) * 0.01
    m_col = torch.randn(n_out, generator=g) * 0.01
    r_row = torch.rand(n_in, generator=g) * 9e-4 + 1e-4
    r_col = torch.rand(n_out, generator=g) * 9e-4 + 1e-4
    x = torch.randn(B, n_in, generator=g)
    want = O.mm8_general_f64(x, codes, r_row, m_row, r_col, m_col)
    packed = ops.pack(codes.cuda())
    got = ops.mm8_packed(x.cuda(), packed, n_in, n_out, r_row.cuda(), m_row.double().cuda(),
                         r_col.cuda(), m_col.cuda()).cpu()
    # float32 accumulation of n_in terms: bound n * 2^-23 * max |partial sum scale|
    scale = (x.abs().double() * r_row.double()) @ codes.double() * r_col.double()
    tol = 2.0 ** -23 * 8 * scale.max()
    err = (got - want).abs().max()
    _say(f"  max err {err:.3e} tol {tol:.3e} |y| {want.abs().max():.3e}")
    assert err <= tol


M16_CASES = [(n_in, n_out, B) for (n_in, n_out) in SHAPES for B in (1, 8)]
M16_CASES += [(96, 40, 3), (130, 77, 5), (768, 50277, 2), (4160, 48, 7), (20480, 32, 8), (64, 16, 1)]


@pytest.mark.parametrize("n_in,n_out,B", M16_CASES)
def test_mm8_m16_general_form(ops, n_in, n_out, B):
    """The matrix-core route of the same product (any B in 1..8, M16 layout): exact integer sums over fp32(x * r_row),
    so it is held to a bound 64 times tighter than the float32-accumulating kernel - what is left is the float32
    rounding of x * r_row itself."""
    _say(f"mm8_m16 in={n_in} out={n_out} B={B}")
    g = torch.Generator().manual_seed(n_in + 3 * n_out + B)
    codes = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8)
    m_row = torch.randn(n_in, generator=g) * 0.01
    m_col = torch.randn(n_out, generator=g) * 0.01
    r_row = torch.rand(n_in, generator=g) * 9e-4 + 1e-4
    r_col = torch.rand(n_out, generator=g) * 9e-4 + 1e-4
    x = torch.randn(B, n_in, generator=g)
    x[0, : n_in // 3] *= 300.0                      # chunks of very different magnitude inside one vector
    want = O.mm8_general_f64(x, codes, r_row, m_row, r_col, m_col)
    p16 = ops.pack_m16(codes.cuda())
    got = ops.mm8_m16(x.cuda(), p16, n_in, n_out, r_row.cuda(), m_row.double().cuda(), r_col.cuda(), m_col.cuda()).cpu()
    scale = (x.abs().double() * r_row.double()) @ codes.double() * r_col.double()
    tol = 2.0 ** -23 * scale.max(dim=1, keepdim=True).values / 8
    err = ((got - want).abs() / tol).max()
    _say(f"  max err / tol {err:.3e}")
    assert err <= 1.0
    # the reference layout (no per-column vectors) against the oracle's mm8_naive with exact accumulation
    got = ops.mm8_m16(x.cuda(), p16, n_in, n_out, r_row.cuda(), m_row.double().cuda()).cpu()
    want = O.mm8_naive(x.double(), codes, r_row, m_row.double(), dtype=torch.float64)
    scale = (x.abs().double() * r_row.double()) @ codes.double()
    assert ((got - want).abs() <= 2.0 ** -23 * scale.max(dim=1, keepdim=True).values / 8).all()


def test_mm8_m16_agrees_with_mm8_packed_and_rejects_bad_arguments(ops):
    from rwkvstic_amd._native import RwkvHipError
    g = torch.Generator().manual_seed(77)
    n_in, n_out = 2560, 2560
    codes = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8).cuda()
    r = (torch.rand(n_in, generator=g) * 9e-4 + 1e-4).cuda()
    m = (torch.randn(n_in, generator=g) * 0.01).double().cuda()
    x = torch.randn(8, n_in, generator=g).cuda()
    a = ops.mm8_packed(x, ops.pack(codes), n_in, n_out, r, m)
    b = ops.mm8_m16(x, ops.pack_m16(codes), n_in, n_out, r, m)
    assert (a - b).abs().max() < 2e-4 * float(b.abs().max())
    # one vector of the eight on its own: the same bits (a vector's digits do not depend on its neighbours)
    b3 = ops.mm8_m16(x[3:4].contiguous(), ops.pack_m16(codes), n_in, n_out, r, m)
    assert torch.equal(b3[0], b[3])
    with pytest.raises(RwkvHipError):
        ops.mm8_m16(torch.zeros(9, n_in, device="cuda"), ops.pack_m16(codes), n_in, n_out, r, m)      # B > 8
    with pytest.raises(RwkvHipError):
        ops.mm8_m16(x, ops.pack_m16(codes), n_in, n_out, r, m, workspace=torch.empty(1024, dtype=torch.uint8, device="cuda"))
    with pytest.raises(ValueError):
        ops.mm8_m16(x, ops.pack_m16(codes)[:1000], n_in, n_out, r, m)


@pytest.mark.parametrize("B", [1, 2, 4])
def test_mm8_packed_reference_form_matches_cpu_path(ops, B):
    """r_col = m_col = None is MM8.forward; compare with the oracle's mm8_naive."""
    W = torch.randn(1000, 384) * 0.02
    c, r, o = O.quantize_matrix(W)
    x = torch.randn(B, 384)
    want = O.mm8_naive(x.double(), c, r, o)
    got = ops.mm8_packed(x.cuda(), ops.pack(c.cuda()), 384, 1000, r.cuda(), o.cuda()).cpu()
    assert (got - want).abs().max() < 2e-5


def test_mm8_packed_rejects_bad_arguments(ops):
    from rwkvstic_amd._native import RwkvHipError
    c = torch.zeros((128, 8), dtype=torch.uint8, device="cuda")
    p = ops.pack(c)
    x = torch.zeros((3, 128), device="cuda")
    r = torch.ones(128, device="cuda"); m = torch.zeros(128, dtype=torch.float64, device="cuda")
    with pytest.raises(RwkvHipError):
        ops.mm8_packed(x, p, 128, 8, r, m)          # B = 3 unsupported
    with pytest.raises(ValueError):
        ops.mm8_packed(x[:1], p[:512], 128, 8, r, m)  # packed too small
    with pytest.raises(TypeError):
        ops.mm8_packed(x[:1].double(), p, 128, 8, r, m)


# ------------------------------------------------------------------ reference-layout operators
@pytest.mark.parametrize("n_in,n_out", [(768, 768), (2560, 2560), (96, 50277), (130, 77)])
def test_mm8_one_reference_semantics(ops, n_in, n_out):
    _say(f"mm8_one in={n_in} out={n_out}")
    g = torch.Generator().manual_seed(n_in * 5 + n_out)
    w = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8)
    r = torch.rand(n_in, generator=g) * 1e-3
    x = torch.randn(n_in, generator=g)
    y0 = torch.randn(n_out, generator=g)
    want = y0.double() + (x.double() * r.double()) @ w.double()
    y = y0.clone().cuda()
    ops.mm8_one(n_in, n_out, x.cuda(), w.cuda(), y, r.cuda())      # accumulates into y
    scale = ((x.abs().double() * r.double()) @ w.double()).max()
    assert (y.cpu().double() - want).abs().max() <= 2.0 ** -23 * 8 * scale + 1e-6 * y0.abs().max()


# 16-byte pieces of rows that start anywhere, the last piece of a row, fewer columns than one piece, slices of 128 rows
# and (from 256 workgroups on) of 256 rows, whole and ragged ones of both
@pytest.mark.parametrize("n_in,n_out,pad", [(1, 1, 0), (127, 15, 3), (128, 16, 0), (129, 17, 5), (256, 127, 1), (257, 129, 0),
                                            (5121, 130, 2), (64, 1100, 7), (2560, 3329, 3), (1800, 4097, 0)])
def test_mm8_one_edges_against_the_float64_product(ops, n_in, n_out, pad):
    _say(f"mm8_one edges in={n_in} out={n_out} pad={pad}")
    g = torch.Generator().manual_seed(n_in * 3 + n_out)
    big = torch.randint(0, 256, (n_in, n_out + pad), generator=g, dtype=torch.uint8)
    x, r, y0 = torch.randn(n_in, generator=g), torch.rand(n_in, generator=g) * 1e-3, torch.randn(n_out, generator=g)
    for dt, eps in ((torch.float32, 2.0 ** -24), (torch.float64, 2.0 ** -53)):
        xd, rd, y = x.to(dt).cuda(), r.to(dt).cuda(), y0.to(dt).cuda()
        ops.mm8_one(n_in, n_out, xd, big.cuda()[:, :n_out], y, rd)
        xr, wd = x.double() * r.double(), big[:, :n_out].double()
        want, mag = y0.double() + xr @ wd, y0.double().abs() + xr.abs() @ wd
        # at most 8 products per lane, 3 + 2 additions in the trees, the slices, the product x * r and y
        steps = 8 + 5 + (n_in + 127) // 128 + 2
        assert ((y.cpu().double() - want).abs() <= steps * eps * mag).all()


# float32 by whole rows: 1024 columns and 128 rows to a workgroup, whole and ragged ones of both, rows that start anywhere, fewer rows
# than the workgroup has wavefronts, three matrices in a call
@pytest.mark.parametrize("n_in,n_out,pad", [(1, 1024, 0), (15, 1023, 2), (128, 1025, 0), (129, 1040, 7), (300, 2047, 1), (1000, 16, 3)])
def test_mm8_by_rows_against_the_float64_product(ops, n_in, n_out, pad):
    _say(f"mm8 by rows in={n_in} out={n_out} pad={pad}")
    g = torch.Generator(device="cuda").manual_seed(n_in * 7 + n_out)
    big = torch.randint(0, 256, (3, n_in, n_out + pad), generator=g, dtype=torch.uint8, device="cuda")
    x, r = torch.randn(n_in, generator=g, device="cuda"), torch.rand(n_in, generator=g, device="cuda") * 1e-3
    y0 = torch.randn(n_out, generator=g, device="cuda")
    z = [y0.clone() for _ in range(3)]
    w = [big[i, :, :n_out] for i in range(3)]
    ops.mm8_three(n_in, n_out, x, x, x, *w, *z, r, r, r)
    for i in range(3):
        y = y0.clone()
        ops.mm8_one(n_in, n_out, x, w[i], y, r)
        assert torch.equal(y, z[i])
        xr, wd = x.double() * r.double(), w[i].double()
        # at most 8 products per lane, 4 additions over the wavefronts, the slices, x * r and y
        steps = 8 + 4 + (n_in + 127) // 128 + 2
        assert ((y.double() - (y0.double() + xr @ wd)).abs() <= steps * 2.0 ** -24 * (y0.double().abs() + xr.abs() @ wd)).all()


# float64: 512 and 1024 rows to a workgroup, the last ones ragged, one row into a further round of 256
@pytest.mark.parametrize("n_in,n_out,pad", [(2049, 8200, 3), (1793, 8321, 0), (5000, 13200, 0), (4097, 16384, 1)])
def test_mm8_float64_of_long_slices_against_the_exact_product(ops, n_in, n_out, pad):
    _say(f"mm8 float64 long slices in={n_in} out={n_out}")
    g = torch.Generator(device="cuda").manual_seed(n_in + n_out)
    big = torch.randint(0, 256, (n_in, n_out + pad), generator=g, dtype=torch.uint8, device="cuda")
    x = torch.randn(n_in, generator=g, device="cuda", dtype=torch.float64)
    r = torch.rand(n_in, generator=g, device="cuda", dtype=torch.float64) * 1e-3
    y0 = torch.randn(n_out, generator=g, device="cuda", dtype=torch.float64)
    y, z = y0.clone(), [y0.clone() for _ in range(3)]
    w = big[:, :n_out]
    ops.mm8_one(n_in, n_out, x, w, y, r)
    ops.mm8_three(n_in, n_out, x, x, x, w, w, w, z[0], z[1], z[2], r, r, r)
    xr, wd = x * r, w.double()
    # at most 32 products per lane, 3 + 2 additions in the trees, the slices, x * r and y on each side
    bound = (2 * (32 + 5 + n_in // 512 + 3)) * 2.0 ** -53 * (y0.abs() + xr.abs() @ wd) + n_in * 2.0 ** -53 * (xr.abs() @ wd)
    assert ((y - (y0 + xr @ wd)).abs() <= bound).all()
    assert all(torch.equal(t, y) for t in z)


# one row more than 65535 slices of 256 rows, in whole cache lines of columns and byte by byte
@pytest.mark.parametrize("n_out", [16, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_mm8_takes_more_rows_than_a_grid_has_slices(ops, n_out, dtype):
    n_in = 65535 * 256 + 1
    _say(f"mm8 in={n_in} out={n_out} {dtype}")
    g = torch.Generator(device="cuda").manual_seed(n_out)
    w = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8, device="cuda")
    # a few thousand rows of +-1/4, the first and the last ones among them: sums of multiples of 1/4 below 2^20 are exact
    rows = torch.unique(torch.cat([torch.randint(0, n_in, (3000,), generator=g, device="cuda"), torch.arange(4, device="cuda"),
                                   torch.arange(n_in - 600, n_in, device="cuda")]))
    x = torch.zeros(n_in, dtype=dtype, device="cuda")
    x[rows] = (torch.randint(0, 2, rows.shape, generator=g, device="cuda") * 2 - 1).to(dtype)
    y = torch.zeros(n_out, dtype=dtype, device="cuda")
    ops.mm8_one(n_in, n_out, x, w, y, torch.full((n_in,), 0.25, dtype=dtype, device="cuda"))
    assert torch.equal(y.double(), (x[rows].double()[:, None] * w[rows].double()).sum(0) * 0.25)


def test_mm8_three_matches_three_mm8_one(ops):
    n_in, n_out = 512, 520
    g = torch.Generator().manual_seed(11)
    ws = [torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8).cuda() for _ in range(3)]
    rs = [(torch.rand(n_in, generator=g) * 1e-3).cuda() for _ in range(3)]
    xs = [torch.randn(n_in, generator=g).cuda() for _ in range(3)]
    y3 = [torch.zeros(n_out, device="cuda") for _ in range(3)]
    y1 = [torch.zeros(n_out, device="cuda") for _ in range(3)]
    ops.mm8_three(n_in, n_out, *xs, *ws, *y3, *rs)
    for i in range(3):
        ops.mm8_one(n_in, n_out, xs[i], ws[i], y1[i], rs[i])
        assert torch.equal(y3[i], y1[i])       # same kernel arithmetic, deterministic


@pytest.mark.parametrize("n_in,n_out", [(768, 768), (130, 77), (2560, 2560), (1000, 50277)])
def test_mm8_one_and_three_float64_instances(ops, n_in, n_out):
    """The `double` branch of the reference's operators (wrapper.cpp:60-77, operators.cu:58-118): x, r, y and the sums
    float64.  Against the float64 dense product at float64 rounding, accumulating into y; three problems in one call
    equal three single calls bit for bit; the float32 instance is left as it was (dtype picks the instance)."""
    _say(f"mm8_one/three f64 in={n_in} out={n_out}")
    g = torch.Generator().manual_seed(n_in * 7 + n_out)
    ws = [torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8) for _ in range(3)]
    rs = [torch.rand(n_in, generator=g, dtype=torch.float64) * 1e-3 for _ in range(3)]
    xs = [torch.randn(n_in, generator=g, dtype=torch.float64) for _ in range(3)]
    y0 = [torch.randn(n_out, generator=g, dtype=torch.float64) for _ in range(3)]
    y1 = [t.clone().cuda() for t in y0]
    y3 = [t.clone().cuda() for t in y0]
    dws = [w.cuda() for w in ws]
    for i in range(3):
        ops.mm8_one(n_in, n_out, xs[i].cuda(), dws[i], y1[i], rs[i].cuda())
        want = y0[i] + (xs[i] * rs[i]) @ ws[i].double()
        scale = ((xs[i].abs() * rs[i]) @ ws[i].double()).max()
        assert (y1[i].cpu() - want).abs().max() <= 2.0 ** -52 * 64 * scale + 1e-15 * y0[i].abs().max()
    ops.mm8_three(n_in, n_out, *[x.cuda() for x in xs], *dws, *y3, *[r.cuda() for r in rs])
    for i in range(3):
        assert torch.equal(y3[i], y1[i])
    with pytest.raises(TypeError):
        ops.mm8_one(n_in, n_out, xs[0].cuda(), dws[0], y1[0].float(), rs[0].cuda())      # mixed types, as wrapper.cpp:58 asserts
    # through the registered operator, as scripted reference code reaches it
    ops.register_torch_ops()
    y = torch.zeros(n_out, dtype=torch.float64, device="cuda")
    torch.ops.rwkv.mm8_one(n_in, n_out, xs[0].cuda(), dws[0], y, rs[0].cuda())
    want = (xs[0] * rs[0]) @ ws[0].double()
    assert (y.cpu() - want).abs().max() <= 2.0 ** -52 * 64 * ((xs[0].abs() * rs[0]) @ ws[0].double()).max()


def test_mm8_one_strided_rows(ops):
    big = torch.randint(0, 256, (64, 1003), dtype=torch.uint8, device="cuda")   # odd stride: byte path
    w = big[:, :1000]
    x = torch.randn(64, device="cuda"); r = torch.rand(64, device="cuda")
    y = torch.zeros(1000, device="cuda")
    ops.mm8_one(64, 1000, x, w, y, r)
    want = (x.double() * r.double()) @ w.double()
    assert (y.double() - want).abs().max() < 1e-2 * 1e-3 * want.abs().max() + 1e-3


def test_torch_ops_registered_with_reference_schema(ops):
    ops.register_torch_ops()
    n_in, n_out = 128, 64
    w = torch.randint(0, 256, (n_in, n_out), dtype=torch.uint8, device="cuda")
    x = torch.randn(n_in, device="cuda"); r = torch.rand(n_in, device="cuda")
    y = torch.zeros(n_out, device="cuda")
    torch.ops.rwkv.mm8_one(n_in, n_out, x, w, y, r)
    assert (y.double() - (x.double() * r.double()) @ w.double()).abs().max() < 1e-2


def _calls(ops):
    """Calls of the published operators, ordinary and odd: (name, arguments).  The last tensors are what they write."""
    g = torch.Generator().manual_seed(5)
    n_in, n_out = 96, 40
    for dt in (torch.float32, torch.float64):
        x, r, y = torch.randn(n_in, generator=g, dtype=dt).cuda(), torch.rand(n_in, generator=g, dtype=dt).cuda(), torch.zeros(n_out, dtype=dt, device="cuda")
        w = torch.randint(0, 256, (n_in, n_out + 8), generator=g, dtype=torch.uint8).cuda()
        yield "mm8_one", (n_in, n_out, x, w[:, :n_out].contiguous(), y, r)
        yield "mm8_one", (n_in, n_out, x, w[:, 3:3 + n_out], y, r)                              # strided rows that start anywhere
        yield "mm8_one", (n_in, n_out, x, w[:, :n_out], y, torch.stack((r, r), 1)[:, 0])         # (a strided r is read as it lies)
        yield "mm8_one", (n_in - 1, n_out, x, w, y, r)                                           # larger tensors than the product
        yield "mm8_one", (n_in, n_out, x.clone().requires_grad_(), w, y, r)
        yield "mm8_one", (n_in, n_out, x[::2], w, y, r)                                          # refused: stride
        yield "mm8_one", (n_in, n_out, x, w.t(), y, r)
        yield "mm8_one", (n_in, n_out, x, w, y[:-1], r)                                          # refused: size
        yield "mm8_one", (n_in, n_out, x, w, y.half(), r)                                        # refused: type
        yield "mm8_one", (0, n_out, x, w, y, r)
        yield "mm8_three", (n_in, n_out, x, x, x, w, w[:, 1:1 + n_out], w, y, y.clone(), y.clone(), r, r, r)
        yield "mm8_three", (n_in, n_out, x, x, x, w, w[:-1], w, y, y.clone(), y.clone(), r, r, r)     # refused: size
        yield "mm8_three", (n_in, n_out, x, x[:-1], x, w, w, w, y, y.clone(), y.clone(), r, r, r)
        yield "mm8_three", (n_in, n_out, x, x, x, w, w, w, y, y.clone(), y.clone()[:-1], r, r, r)
        yield "mm8_three", (n_in, n_out, x, x, x, w, w, w, y, y.clone(), y.clone(), r[1:], r, r)
        yield "mm8_one", (n_in, n_out, x, w, y, r.new_ones(1).expand(n_in))                              # refused: as many values, less memory
        yield "mm8_one", (n_in, n_out, x, w, y.new_ones(1, 1).expand(1, n_out), r)
    f = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64).cuda()
    wkv = lambda T, C: (2, T, C, -f(C), f(C), f(2, T, C), f(2, T, C), f(2, T, C), f(2, C), f(2, C) + 0.5, f(2, C))
    yield "wkv_forward", wkv(3, 5)
    yield "wkv_forward", wkv(20, 33)
    yield "wkv_forward", wkv(3, 5)[:5] + (f(5, 6).t(),) + wkv(3, 5)[6:]
    yield "wkv_forward", (2, 4, 5) + wkv(3, 5)[3:]


def test_published_operators_do_what_the_functions_do(ops):
    """Results, and what is refused with which exception: the operators' native side leaves odd calls to the functions."""
    ops.register_torch_ops()
    for i, (name, args) in enumerate(_calls(ops)):
        print(f"operator call {i}: {name}", flush=True)
        seen = []
        for fn in (getattr(ops, name), getattr(torch.ops.rwkv, name)):
            mine = [a.detach().clone(memory_format=torch.preserve_format).requires_grad_(a.requires_grad)
                    if isinstance(a, torch.Tensor) and a.is_contiguous() else a for a in args]
            try:
                fn(*mine)
            except Exception as e:
                seen.append((type(e), str(e)))
            else:
                seen.append([a.detach().cpu() for a in mine if isinstance(a, torch.Tensor)])
        if isinstance(seen[0], tuple):
            assert seen[0] == seen[1], (i, seen)
        else:
            assert not isinstance(seen[1], tuple), (i, seen[1])
            assert all(torch.equal(a, b) for a, b in zip(*seen)), i


# ------------------------------------------------------------------ WKV
def _wkv_case(B, T, C, seed, lo=-8.0):
    g = torch.Generator().manual_seed(seed)
    k = torch.randn(B, T, C, generator=g)
    v = torch.randn(B, T, C, generator=g)
    w = -torch.exp(torch.rand(C, generator=g) * (1.0 - lo) + lo)
    u = torch.rand(C, generator=g) * 2 - 1
    return w, u, k, v


def _check_wkv_f32(ops, B, T, C, seed):
    w, u, k, v = _wkv_case(B, T, C, seed)
    aa = torch.zeros(B, C); bb = torch.zeros(B, C); pp = torch.full((B, C), -1e38)
    d = lambda t: t.cuda()
    aa_d, bb_d, pp_d = d(aa), d(bb), d(pp)
    y = ops.wkv_f32(d(w), d(u), d(k), d(v), aa_d, bb_d, pp_d).cpu()
    for b in range(B):
        yr, ar, br, _ = O.wkv_naive(w.double(), u.double(), k[b].double(), v[b].double(),
                                    aa[b].double(), bb[b].double(), pp[b].double())
        assert (y[b].double() - yr).abs().max() < 1e-4 * max(1.0, float(yr.abs().max()))
        an, bn = O.state_naive_from_stable(aa_d[b].cpu(), bb_d[b].cpu(), pp_d[b].cpu())
        # bb is a positive sum; aa is a signed sum of the same weights times v ~ N(0,1)
        assert ((bn - br).abs() <= 1e-4 * br).all()
        assert ((an - ar).abs() <= 1e-4 * torch.maximum(ar.abs(), br)).all()


def test_wkv_f32_small(ops):
    _say("wkv_f32 B=2 T=37 C=130")
    _check_wkv_f32(ops, 2, 37, 130, seed=3)


def test_wkv_f32_isolated_workload(ops):
    _say("wkv_f32 B=8 T=1024 C=2560")
    _check_wkv_f32(ops, 8, 1024, 2560, seed=2)


def test_wkv_f32_split_invariance_and_large_k(ops):
    """Carrying the state across two calls equals one call; k up to +-60 must not overflow float32."""
    w, u, k, v = _wkv_case(1, 64, 64, seed=9)
    k = k * 20
    d = lambda t: t.cuda()
    s1 = [torch.zeros(1, 64).cuda(), torch.zeros(1, 64).cuda(), torch.full((1, 64), -1e38).cuda()]
    y_all = ops.wkv_f32(d(w), d(u), d(k), d(v), *s1)
    s2 = [torch.zeros(1, 64).cuda(), torch.zeros(1, 64).cuda(), torch.full((1, 64), -1e38).cuda()]
    ya = ops.wkv_f32(d(w), d(u), d(k[:, :20].contiguous()), d(v[:, :20].contiguous()), *s2)
    yb = ops.wkv_f32(d(w), d(u), d(k[:, 20:].contiguous()), d(v[:, 20:].contiguous()), *s2)
    # the exponent is float64 inside a call and rounded to float32 at the call boundary
    assert torch.allclose(torch.cat([ya, yb], 1), y_all, rtol=2e-5, atol=2e-5)
    assert torch.isfinite(y_all).all()
    yr = O.wkv_stable(w.double(), u.double(), k[0].double(), v[0].double(),
                      torch.zeros(64).double(), torch.zeros(64).double(), torch.full((64,), -1e38).double())[0]
    assert (y_all[0].cpu().double() - yr).abs().max() < 1e-4 * max(1.0, float(yr.abs().max()))


@pytest.mark.parametrize("T", [256, 333, 1000])
def test_wkv_f32_long_sequences_carry_a_state_in_and_out(ops, T):
    """Sequences of 256 steps and more run as a two-pass scan inside a workgroup (ragged last chunks at 333 and
    1000): a state carried in from a first call, the outputs and the state carried out against the float64
    recurrence over both calls; large |k| must not overflow."""
    _say(f"wkv_f32 scan T={T}")
    B, C, T0 = 3, 96, 40
    w, u, k, v = _wkv_case(B, T0 + T, C, seed=11)
    k = k * 8
    d = lambda t: t.cuda()
    st = [torch.zeros(B, C).cuda(), torch.zeros(B, C).cuda(), torch.full((B, C), -1e38).cuda()]
    ya = ops.wkv_f32(d(w), d(u), d(k[:, :T0].contiguous()), d(v[:, :T0].contiguous()), *st)
    yb = ops.wkv_f32(d(w), d(u), d(k[:, T0:].contiguous()), d(v[:, T0:].contiguous()), *st)
    y = torch.cat([ya, yb], 1).cpu().double()
    assert torch.isfinite(y).all()
    for b in range(B):
        z = torch.zeros(C).double()
        yr, ar, br, _ = O.wkv_naive(w.double(), u.double(), k[b].double(), v[b].double(), z, z.clone(), torch.full((C,), -1e38).double())
        assert (y[b] - yr).abs().max() < 1e-4 * max(1.0, float(yr.abs().max()))
        ys, a_s, b_s, p_s = O.wkv_stable(w.double(), u.double(), k[b].double(), v[b].double(), z, z.clone(), torch.full((C,), -1e38).double())
        # the state in its shifted form: aa e^pp and bb e^pp are what the next call continues from
        got_a, got_b, got_p = st[0][b].cpu().double(), st[1][b].cpu().double(), st[2][b].cpu().double()
        scale = torch.exp(got_p - p_s)
        assert ((got_b * scale - b_s).abs() <= 1e-4 * b_s.abs()).all()
        assert ((got_a * scale - a_s).abs() <= 1e-4 * torch.maximum(a_s.abs(), b_s.abs())).all()


@pytest.mark.parametrize("T", [300, 1000])
def test_wkv_f32_one_read_scan_with_ragged_blocks_and_a_carried_state(ops, T):
    """With 512 and more groups of 32 channels the scan keeps each chunk's k and v in registers between its two passes
    and reads them once (blocks of 128 steps; 300 and 1000 end inside a block and inside a chunk): outputs and the
    state carried out, after a state carried in from a first call, against the float64 recurrence; large |k|."""
    _say(f"wkv_f32 one-read scan T={T}")
    B, C, T0 = 8, 2048, 30
    w, u, k, v = _wkv_case(B, T0 + T, C, seed=21)
    k = k * 6
    d = lambda t: t.cuda()
    st = [torch.zeros(B, C).cuda(), torch.zeros(B, C).cuda(), torch.full((B, C), -1e38).cuda()]
    ya = ops.wkv_f32(d(w), d(u), d(k[:, :T0].contiguous()), d(v[:, :T0].contiguous()), *st)
    yb = ops.wkv_f32(d(w), d(u), d(k[:, T0:].contiguous()), d(v[:, T0:].contiguous()), *st)
    y = torch.cat([ya, yb], 1).cpu().double()
    assert torch.isfinite(y).all()
    for b in (0, 3, 7):
        z = torch.zeros(C).double()
        ys, a_s, b_s, p_s = O.wkv_stable(w.double(), u.double(), k[b].double(), v[b].double(), z, z.clone(), torch.full((C,), -1e38).double())
        assert (y[b] - ys).abs().max() < 1e-4 * max(1.0, float(ys.abs().max()))
        got_a, got_b, got_p = st[0][b].cpu().double(), st[1][b].cpu().double(), st[2][b].cpu().double()
        scale = torch.exp(got_p - p_s)
        assert ((got_b * scale - b_s).abs() <= 1e-4 * b_s.abs()).all()
        assert ((got_a * scale - a_s).abs() <= 1e-4 * torch.maximum(a_s.abs(), b_s.abs())).all()


def test_wkv_forward_f64_reference_convention(ops):
    """Drop-in for torch.ops.rwkv.wkv_forward: naive state in/out, pp untouched."""
    B, T, C = 1, 50, 96
    w, u, k, v = _wkv_case(B, T, C, seed=4)
    w, u, k, v = (t.double() for t in (w, u, k, v))
    aa = torch.rand(C).double(); bb = torch.rand(C).double() + 0.5; pp = torch.full((C,), -1e30).double()
    yr, ar, br, pr = O.wkv_naive(w, u, k[0], v[0], aa, bb, pp)
    d = lambda t: t.cuda()
    aa_d, bb_d, pp_d = d(aa.clone()), d(bb.clone()), d(pp.clone())
    y = torch.empty(T, C, dtype=torch.float64, device="cuda")
    ops.wkv_forward(1, T, C, d(w), d(u), d(k[0].contiguous()), d(v[0].contiguous()), y, aa_d, bb_d, pp_d)
    assert torch.allclose(y.cpu(), yr, rtol=1e-11, atol=1e-12)
    assert torch.allclose(aa_d.cpu(), ar, rtol=1e-10) and torch.allclose(bb_d.cpu(), br, rtol=1e-10)
    assert torch.equal(pp_d.cpu(), pp)
    # from the empty state too
    z = torch.zeros(C).double()
    yr, ar, br, _ = O.wkv_naive(w, u, k[0], v[0], z, z.clone(), pp)
    aa_d, bb_d = d(z.clone()), d(z.clone())
    ops.wkv_forward(1, T, C, d(w), d(u), d(k[0].contiguous()), d(v[0].contiguous()), y, aa_d, bb_d, pp_d)
    assert torch.allclose(y.cpu(), yr, rtol=1e-11, atol=1e-12)
    assert torch.allclose(bb_d.cpu(), br, rtol=1e-10)


# the serial kernel and both scan forms, at the edges of their chunks (8 steps) and blocks (64 and 256 steps)
@pytest.mark.parametrize("T", [1, 11, 12, 63, 64, 65, 255, 256, 257, 600])
@pytest.mark.parametrize("B,C", [(1, 32), (3, 33)])
def test_wkv_forward_f64_any_length(ops, B, T, C):
    _wkv_f64_case(ops, B, T, C)


# both sides of the lengths from which so many channels are scanned, and more channels than are scanned at all
@pytest.mark.parametrize("B,C,T", [(50, 640, 31), (50, 640, 32), (50, 640, 79), (50, 640, 80), (100, 1001, 65), (7, 160, 12)])
def test_wkv_forward_f64_of_many_channels(ops, B, C, T):
    _wkv_f64_case(ops, B, T, C)


# the widths of the scan's workgroups: 8, 16, 32 and 16 channels, at the edges of the rule and with a ragged last one
@pytest.mark.parametrize("B,C,T", [(1, 2048, 65), (1, 2049, 65), (2, 1030, 257), (1, 4096, 100), (1, 4097, 100), (8, 1024, 70), (3, 2731, 70)])
def test_wkv_forward_f64_workgroup_widths(ops, B, C, T):
    _wkv_f64_case(ops, B, T, C)


def _wkv_f64_case(ops, B, T, C):
    _say(f"wkv_forward f64 B={B} T={T} C={C}")
    w, u, k, v = (t.double() for t in _wkv_case(B, T, C, seed=T + C))
    g = torch.Generator().manual_seed(T)
    aa, bb = torch.randn(B, C, generator=g).double(), torch.rand(B, C, generator=g).double() + 0.5
    aa[0, :3], bb[0, :3] = 0.0, 0.0                     # three empty channels among the others
    pp = torch.full((B, C), -1e30).double()
    y, ad, bd, pd = torch.empty(B, T, C, dtype=torch.float64, device="cuda"), aa.cuda(), bb.cuda(), pp.cuda()
    ops.wkv_forward(B, T, C, w.cuda(), u.cuda(), k.cuda(), v.cuda(), y, ad, bd, pd)
    for b in range(B):
        yr, ar, br, _ = O.wkv_naive(w, u, k[b], v[b], aa[b], bb[b], pp[b])
        assert torch.allclose(y[b].cpu(), yr, rtol=1e-11, atol=1e-12)
        assert torch.allclose(ad[b].cpu(), ar, rtol=1e-10, atol=1e-12) and torch.allclose(bd[b].cpu(), br, rtol=1e-10)
    assert torch.equal(pd.cpu(), pp)


def test_argmax_first_maximum(ops):
    x = torch.randn(50277, dtype=torch.float64)
    x[40000] = 9.0; x[123] = 9.0
    assert int(ops.argmax(x.cuda())) == 123


def test_pack_m16_round_trip(ops):
    for n_in, n_out in [(64, 16), (130, 77), (2560, 2560)]:
        c = torch.randint(0, 256, (n_in, n_out), dtype=torch.uint8, device="cuda")
        p = ops.pack_m16(c)
        assert torch.equal(ops.unpack_m16(p, n_in, n_out), c)
    # block 0, lane 16*g + n, byte i  <->  codes[16*g + i][n] - 128
    c = torch.arange(64 * 16, dtype=torch.int64).reshape(64, 16).remainder(256).to(torch.uint8).cuda()
    p = ops.pack_m16(c).cpu().reshape(64, 16)
    for lane in (0, 5, 17, 63):
        g, n = divmod(lane, 16)
        want = (c[16 * g:16 * g + 16, n].cpu().to(torch.int16) - 128).to(torch.int8)
        assert torch.equal(p[lane].view(torch.int8), want)


# the last two run the 160-column workgroup variant (320 general workgroups would make 1.25 per compute unit),
# with ragged rows, ragged columns and a contraction that ends inside a round of the pipeline
@pytest.mark.parametrize("T,K,N", [(1, 64, 16), (5, 256, 100), (64, 2560, 2560), (130, 2560, 10240),
                                   (33, 10240, 2560), (8, 2560, 50277), (1000, 192, 2560), (1024, 320, 2500),
                                   (3, 20544, 32),      # a few long rows: the two-launch quantiser
                                   (4, 8320, 48),       # the same with parts that have to be rounded up to whole groups of 16 values
                                   (9, 20544, 32),      # rows too long for the register-resident quantiser
                                   (20, 2560, 2560), (32, 640, 5000),    # 9..32 rows: the few-row variant with LDS staging
                                   # 769..960 rows on a long contraction: the 160-column workgroups (208 of them)
                                   (800, 2560, 2560), (900, 2560, 5120),
                                   # the 128-column workgroups with the contraction split (80 workgroups x 2,
                                   # 20 x 4: integer slices added by the tail kernel), ragged rows
                                   (250, 2560, 2560), (60, 10240, 2560)])
def test_gemm8_matches_fp64_dense(ops, T, K, N):
    """Prompt GEMM (matmul.py:56-57 without its bfloat16 rounding) against the float64 dense product."""
    g = torch.Generator().manual_seed(T * 7 + K + N)
    w = torch.randn(N, K, generator=g) * 0.02
    codes, rng, off = O.quantize_matrix(w)
    x = torch.randn(T, K, generator=g, dtype=torch.float64)
    x[0, : K // 2] *= 50.0                                    # rows with very different scales
    want = O.mm8_naive(x, codes, rng, off, dtype=torch.float64)
    dev = "cuda"
    p16 = ops.pack_m16(codes.to(dev))
    got = ops.gemm8(x.to(dev), p16, rng.to(dev), off.to(dev), K, N).cpu()
    bound = ((x.abs() * rng.double()) @ codes.double()).max(dim=1, keepdim=True).values
    err = ((got - want).abs() / bound).max().item()
    print(f"gemm8 T={T} K={K} N={N}: max err / sum|terms| = {err:.2e}", flush=True)
    assert err < 2e-7                                         # float32 rounding of x*range, nothing else


# grids that leave compute units idle: 80 columns to a workgroup.  Ragged rows, columns and column blocks, fewer contraction blocks than
# the ring has buffers, XCDs that share out the columns (up to 7 row blocks) and the rows
@pytest.mark.parametrize("T,K,N", [(300, 2560, 2560), (200, 64, 4096), (130, 128, 5000), (400, 704, 2502), (520, 192, 1200), (512, 320, 2560)])
def test_gemm8_of_narrow_workgroups_matches_fp64_dense(ops, T, K, N):
    import ctypes
    from rwkvstic_amd import _native
    plan, tot = (ctypes.c_int * 4)(), ctypes.c_size_t()
    _native.check(_native.lib().rwkv_gemm8_plan(T, K, N, 1, plan, ctypes.byref(tot)))
    assert (plan[0], plan[1], plan[3]) == (3, -(-N // 80), 1)
    test_gemm8_matches_fp64_dense(ops, T, K, N)


# at most 8 rows: both sides of the column tiles at which the kernel changes its shape (256 | 320 | 512 | 1280),
# fewer blocks than wavefronts, one block past a round, a split contraction
@pytest.mark.parametrize("T,K,N", [(1, 64, 16), (8, 17 * 64, 4096), (8, 17 * 64, 4100), (3, 192, 5120), (5, 41 * 64, 5121), (4, 448, 8192),
                                   (8, 41 * 64, 8200), (8, 192, 20480), (7, 25 * 64, 20490), (6, 49 * 64, 4096), (8, 81 * 64, 256),
                                   (2, 1025 * 64, 20),
                                   # 9 to 32 rows of small matrices: every count of M-tiles, tiles (256 | 320 | 512 | 1280) and
                                   # contractions (blocks times M-tiles 200 | 700, 400) on both sides of the rules' edges
                                   (9, 64, 16), (12, 17 * 64, 4100), (13, 50 * 64, 4112), (16, 50 * 64, 4112), (16, 51 * 64, 4112), (10, 100 * 64, 8192),
                                   (16, 175 * 64, 4096), (15, 176 * 64, 4096), (11, 33 * 64, 8200), (14, 5 * 64, 20480), (9, 6 * 64, 20490),
                                   (17, 64, 16), (20, 80 * 64, 4096), (24, 66 * 64, 4097), (25, 50 * 64, 8192), (32, 50 * 64, 8192), (32, 51 * 64, 8192),
                                   (29, 17 * 64, 8193), (32, 64, 50), (21, 33 * 64, 4100)])
def test_few_row_products_match_fp64_dense(ops, T, K, N):
    g = torch.Generator().manual_seed(T * 7 + K + N)
    codes = torch.randint(0, 256, (K, N), generator=g, dtype=torch.uint8)
    rng, off = torch.rand(K, generator=g) * 1e-3, torch.randn(K, generator=g, dtype=torch.float64) * 0.01
    x = torch.randn(T, K, generator=g, dtype=torch.float64)
    x[0, : K // 2] *= 50.0
    xr = (x * rng.double()).float().double()                 # what the kernel is given to multiply, rounded once
    want = (xr @ codes.double()) + (x @ off)[:, None]
    p16 = ops.pack_m16(codes.cuda())
    got = ops.gemm8(x.cuda(), p16, rng.cuda(), off.cuda(), K, N).cpu()
    # fixed point of 30 bits below a row's largest |xr| (half a unit each, codes up to 255), float64 beyond that
    bound = K * 255 * xr.abs().max(dim=1, keepdim=True).values * 2.0 ** -30 + 1e-12 * (x.abs() @ off.abs())[:, None]
    print(f"few-row product T={T} K={K} N={N}: max err / bound {((got - want).abs() / bound).max():.2e}", flush=True)
    assert ((got - want).abs() <= bound).all()


def test_gemm8_rows_do_not_depend_on_batching(ops):
    """Integer accumulation: a row's result is bit-identical whether the contraction is split (few rows)
    or not (many rows), and wherever the row sits in its tile."""
    g = torch.Generator().manual_seed(3)
    K, N = 2560, 2560
    w = torch.randn(N, K, generator=g) * 0.02
    codes, rng, off = O.quantize_matrix(w)
    x = torch.randn(1024, K, generator=g, dtype=torch.float64).cuda()
    p16 = ops.pack_m16(codes.cuda())
    wide = ops.gemm8(x, p16, rng.cuda(), off.cuda(), K, N)            # 160-column workgroups
    full = ops.gemm8(x[:300].contiguous(), p16, rng.cuda(), off.cuda(), K, N)    # 128-column workgroups
    few = ops.gemm8(x[37:40].contiguous(), p16, rng.cuda(), off.cuda(), K, N)    # few-row variant, split contraction
    assert torch.equal(full[37:40], few) and torch.equal(wide[:300], full)
