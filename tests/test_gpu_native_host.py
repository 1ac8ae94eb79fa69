"""The native host side of the operators (csrc/rwkv_torch.cpp): what it does with the answers of the library, checked with
entry points bound to functions of the test in place of the library's, so that nothing wrong is ever launched."""
import contextlib
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from rwkvstic_amd import ops as _ops
    _ops.register_torch_ops()
    return _ops


@contextlib.contextmanager
def _bound(**entries):
    """The host side with some of its entry points replaced by the addresses given."""
    from rwkvstic_amd import _native as N
    own = {n: C.cast(getattr(N.lib(), n), C.c_void_p).value for n in N.EXPORTS}
    N.host().bind({**own, **entries})
    try:
        yield
    finally:
        N.host().bind(own)


def _calls(ops):
    """Each operator once: (library entry, call, the tensors it writes)."""
    g = torch.Generator().manual_seed(1)
    n_in, n_out = 256, 48
    codes = torch.randint(0, 256, (n_in, n_out), generator=g, dtype=torch.uint8).cuda()
    for dt, suffix in ((torch.float32, ""), (torch.float64, "_f64")):
        x, r = torch.randn(n_in, generator=g, dtype=dt).cuda(), torch.rand(n_in, generator=g, dtype=dt).cuda()
        ys = [torch.randn(n_out, generator=g, dtype=dt).cuda() for _ in range(4)]
        yield "rwkv_mm8_one" + suffix, lambda: torch.ops.rwkv.mm8_one(n_in, n_out, x, codes, ys[0], r), ys[:1]
        yield "rwkv_mm8_three" + suffix, lambda: torch.ops.rwkv.mm8_three(n_in, n_out, x, x, x, codes, codes, codes, *ys[1:], r, r, r), ys[1:]
    for dt, entry in ((torch.float64, "rwkv_wkv_forward_f64"), (torch.float32, "rwkv_wkv_f32")):
        f = lambda *s: torch.rand(*s, generator=g, dtype=dt).cuda()
        w, u, k, v, y = -f(32), f(32), f(2, 5, 32), f(2, 5, 32), f(2, 5, 32)
        state = [f(2, 32), f(2, 32) + 0.5, f(2, 32)]
        if dt == torch.float64:
            yield entry, lambda: torch.ops.rwkv.wkv_forward(2, 5, 32, w, u, k, v, y, *state), state + [y]
        else:
            yield entry, lambda: ops.wkv_f32(w, u, k, v, *state), state
    x, r, m = torch.randn(2, n_in, generator=g).cuda(), torch.rand(n_in, generator=g).cuda(), torch.randn(n_in, generator=g).double().cuda()
    y = torch.randn(2, n_out, generator=g).double().cuda()
    p, p16 = ops.pack(codes), ops.pack_m16(codes)
    yield "rwkv_mm8_packed", lambda: ops.mm8_packed(x, p, n_in, n_out, r, m, out=y), [y]
    yield "rwkv_mm8_m16", lambda: ops.mm8_m16(x, p16, n_in, n_out, r, m, out=y), [y]


def test_an_error_of_the_library_is_raised_and_nothing_is_done_again(ops):
    """A library that answers RWKV_ERR_HIP may have launched all the same, so the call is not repeated by other means."""
    from rwkvstic_amd import _native as N
    for entry, call, written in _calls(ops):
        print(f"error from {entry}", flush=True)
        before, seen = [t.clone() for t in written], []
        fails = C.CFUNCTYPE(C.c_int)(lambda: seen.append(1) or -5)
        with _bound(**{entry: C.cast(fails, C.c_void_p).value}):
            with pytest.raises(N.RwkvHipError) as e:
                call()
        torch.cuda.synchronize()
        assert e.value.code == -5 and len(seen) == 1, entry
        assert all(torch.equal(a, b) for a, b in zip(before, written)), entry


def test_an_error_left_by_another_hip_call_does_not_repeat_an_operator(ops):
    """The same from the other end: a HIP call of this thread has failed (an allocation of 2^60 bytes) and nobody has read
    its error, which the library then reports after its own launch.  Each operator raises, and has run at most once."""
    from rwkvstic_amd import _native as N
    L = N.lib()
    at = C.c_void_p()
    for entry, call, written in _calls(ops):
        print(f"error left before {entry}", flush=True)
        start = [t.clone() for t in written]
        call()
        torch.cuda.synchronize()
        once = [t.clone() for t in written]
        for t, b in zip(written, start):
            t.copy_(b)
        torch.cuda.synchronize()
        assert L.hipMalloc(C.byref(at), C.c_size_t(1 << 60)) != 0
        try:
            call()
        except N.RwkvHipError as e:
            assert e.code == -5
        finally:
            L.hipGetLastError()
        torch.cuda.synchronize()
        for t, a, b in zip(written, start, once):
            assert torch.equal(t, a) or torch.equal(t, b), entry


def test_other_threads_run_while_a_launch_waits(ops):
    """A launch waits where the stream's queue is full.  poll(0, 0, ms) stands for one that does: of no vectors of 300 values (or
    no sequences of 300 steps) on the default stream, the entries' first arguments are just that."""
    import threading
    import time
    ms, f = 300, lambda *s, dt=torch.float32: torch.zeros(*s, dtype=dt, device="cuda")
    codes = torch.zeros(ms, 16, dtype=torch.uint8, device="cuda")
    args = f(ms), f(ms, dt=torch.float64)
    calls = {"rwkv_mm8_packed": lambda p=ops.pack(codes): ops.mm8_packed(f(0, ms), p, ms, 16, *args),
             "rwkv_mm8_m16": lambda p=ops.pack_m16(codes): ops.mm8_m16(f(0, ms), p, ms, 16, *args),
             "rwkv_wkv_f32": lambda: ops.wkv_f32(f(4), f(4), f(0, ms, 4), f(0, ms, 4), f(0, 4), f(0, 4), f(0, 4))}
    assert torch.cuda.current_stream().cuda_stream == 0
    poll = C.cast(C.CDLL(None).poll, C.c_void_p).value
    for entry, call in calls.items():
        rounds, stop = [0], threading.Event()

        def count():
            while not stop.wait(0.001):
                rounds[0] += 1

        t = threading.Thread(target=count)
        t.start()
        try:
            with _bound(**{entry: poll}):
                before, start = rounds[0], time.monotonic()
                call()
                took, ran = time.monotonic() - start, rounds[0] - before
        finally:
            stop.set()
            t.join()
        print(f"{entry}: {took:.3f} s, {ran} rounds of another thread", flush=True)
        assert took >= ms * 1e-3 and ran >= 50, entry


@pytest.mark.parametrize("native", [True, False])
def test_products_of_two_threads_on_two_streams(ops, native):
    """Each call has scratch of its own: threads that multiply at the same time, with products of several workgroup rows whose
    partial sums go through it, get what each gets alone; with the native side, and through the Python functions."""
    import threading
    g = torch.Generator(device="cuda").manual_seed(8)
    fns = torch.ops.rwkv if native else ops
    work = []
    for n_in, n_out, dt in ((4096, 1024, torch.float32), (2560, 1536, torch.float64)):
        x, r = torch.randn(n_in, generator=g, device="cuda").to(dt), torch.rand(n_in, generator=g, device="cuda").to(dt)
        codes = torch.randint(0, 256, (n_in, n_out), generator=g, device="cuda", dtype=torch.uint8)
        rows = torch.randn(24, n_in, generator=g, device="cuda").double()
        work.append((n_in, n_out, x, codes, torch.zeros(n_out, device="cuda", dtype=dt), r, rows, ops.pack_m16(codes), r.float(), r.double()))

    def run(n_in, n_out, x, w, y, r, rows, w16, rng, off):
        three, products = [torch.zeros_like(y) for _ in range(3)], []
        for _ in range(100):
            fns.mm8_one(n_in, n_out, x, w, y, r)
            fns.mm8_three(n_in, n_out, x, x, x, w, w, w, *three, r, r, r)
            products.append(ops.gemm8(rows, w16, rng, off, n_in, n_out))
        return [y, *three, *products]

    want = [[t.clone() for t in run(*a)] for a in work]
    for a in work:
        a[4].zero_()
    torch.cuda.synchronize()
    # both streams wait for a long product, so that their calls are queued by then and run at the same time
    wide = torch.randn(8192, 8192, device="cuda")
    for _ in range(10):
        wide = torch.mm(wide, wide)
    queued = torch.cuda.Event()
    queued.record()
    got, errors = [None, None], []

    def thread(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                queued.wait()
                got[i] = run(*work[i])
                torch.cuda.current_stream().synchronize()
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=thread, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i in range(2):
        assert all(torch.equal(a, b) for a, b in zip(want[i], got[i])), i


def test_scratch_of_a_recorded_product_is_not_given_back(ops):
    """A graph that holds an operator call writes its scratch whenever it is replayed, also after a larger product has been
    recorded: nobody else may have been given that memory."""
    g = torch.Generator(device="cuda").manual_seed(9)

    def product(n_in, n_out):
        x, r = torch.randn(n_in, generator=g, device="cuda"), torch.rand(n_in, generator=g, device="cuda")
        w = torch.randint(0, 256, (n_in, n_out), generator=g, device="cuda", dtype=torch.uint8)
        return n_in, n_out, x, w, torch.zeros(n_out, device="cuda"), r

    def record(a):
        graph, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=st):
            torch.ops.rwkv.mm8_one(*a)
        return graph

    def buffers():
        return [b for kept in ops._scratch.values() for b in (kept if isinstance(kept, list) else [kept])]

    ops._scratch.clear()
    small, large = product(4096, 1024), product(8192, 16384)
    want = torch.zeros_like(small[4])
    torch.ops.rwkv.mm8_one(*small[:4], want, small[5])
    graphs = [record(small)]
    at, size = buffers()[0].data_ptr(), buffers()[0].numel()
    graphs.append(record(large))
    assert any(b.data_ptr() == at for b in buffers()), "the first recording's scratch was given back"
    assert len(buffers()) == 2 and max(b.numel() for b in buffers()) >= 2 * size
    for i in range(3):
        for a, graph in zip((small, large), graphs):
            a[4].zero_()
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(small[4], want), f"replay {i}"
