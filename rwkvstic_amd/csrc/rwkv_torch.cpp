// Host side of the operator calls, native: torch.ops.rwkv.* (reference src/rwkvstic/agnostic/backends/cuda/wrapper.cpp:45-141)
// and the stand-alone products and recurrence of rwkvstic_amd.ops.  A call checks its tensors, takes its workspace from torch's
// allocator (so that it belongs to the stream the call runs on) and hands device pointers to librwkv_hip.so.
//
// What bounds these calls is the host: a matrix of the 3B shape is 10 us of kernels, and a call that goes through Python
// (dispatcher to interpreter, checks, ctypes) takes 16.
//
// An argument that does not fit is left to the Python function of the same name, which raises what it always raised.  Only
// arguments are: what the library reports is raised here, since it may report an error after it has launched (one that an
// earlier HIP call of the thread left behind), and the operators write in place: a second call would add y twice.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <map>
#include <string>
#include <vector>

#include "../../include/rwkv_hip.h"

namespace {

// Entry points of the library that the Python side has loaded (it decides which file that is).
struct Entries {
    decltype(&rwkv_mm8_workspace_bytes) mm8_workspace_bytes, mm8_f64_workspace_bytes;
    decltype(&rwkv_mm8_one) mm8_one;
    decltype(&rwkv_mm8_one_f64) mm8_one_f64;
    decltype(&rwkv_mm8_three) mm8_three;
    decltype(&rwkv_mm8_three_f64) mm8_three_f64;
    decltype(&rwkv_wkv_forward_f64) wkv_forward_f64;
    decltype(&rwkv_packed_bytes) packed_bytes, packed_m16_bytes;
    decltype(&rwkv_mm8_packed) mm8_packed;
    decltype(&rwkv_mm8_m16_workspace_bytes) mm8_m16_workspace_bytes;
    decltype(&rwkv_mm8_m16) mm8_m16;
    decltype(&rwkv_wkv_f32) wkv_f32;
} lib;

void bind(const std::map<std::string, uintptr_t> &at) {
#define BIND(field, name) lib.field = reinterpret_cast<decltype(lib.field)>(at.at(#name))
    BIND(mm8_workspace_bytes, rwkv_mm8_workspace_bytes); BIND(mm8_f64_workspace_bytes, rwkv_mm8_f64_workspace_bytes);
    BIND(mm8_one, rwkv_mm8_one); BIND(mm8_one_f64, rwkv_mm8_one_f64);
    BIND(mm8_three, rwkv_mm8_three); BIND(mm8_three_f64, rwkv_mm8_three_f64);
    BIND(wkv_forward_f64, rwkv_wkv_forward_f64);
    BIND(packed_bytes, rwkv_packed_bytes); BIND(packed_m16_bytes, rwkv_packed_m16_bytes);
    BIND(mm8_packed, rwkv_mm8_packed);
    BIND(mm8_m16_workspace_bytes, rwkv_mm8_m16_workspace_bytes); BIND(mm8_m16, rwkv_mm8_m16);
    BIND(wkv_f32, rwkv_wkv_f32);
#undef BIND
}

using Stream = c10::hip::HIPStream;
Stream current() { return c10::hip::getCurrentHIPStream(); }
rwkv_stream_t handle(const Stream &st) { return reinterpret_cast<rwkv_stream_t>(st.stream()); }

// A recorded call keeps its scratch for as long as it is replayed: the buffer the Python side holds on to.
bool recording(const Stream &st) {
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st.stream(), &s) != hipSuccess) { (void)hipGetLastError(); return true; }
    return s != hipStreamCaptureStatusNone;
}

// What the library answers to a call: RwkvHipError with its text for anything but RWKV_OK.
void check(int code) {
    if (code == RWKV_OK) return;
    pybind11::gil_scoped_acquire gil;
    pybind11::module_::import("rwkvstic_amd._native").attr("check")(code);
}

// Whether a call on this stream may take scratch from the allocator: that belongs to x's device, and only where the stream does too may
// it be handed out again after the call.
bool scratch_fits(const Stream &st, const at::Tensor &x) { return x.is_cuda() && x.get_device() == st.device_index() && !recording(st); }

at::Tensor bytes(size_t n, const at::Tensor &like) {
    return at::empty({static_cast<int64_t>(n > 0 ? n : 1)}, like.options().dtype(at::kByte));
}

bool on_gpu(const at::Tensor &t, at::ScalarType dt) { return t.defined() && t.is_cuda() && t.scalar_type() == dt && !t.requires_grad(); }
bool vec(const at::Tensor &t, at::ScalarType dt) { return on_gpu(t, dt) && t.dim() == 1 && t.stride(0) == 1; }
bool codes(const at::Tensor &w, int64_t n, int64_t m) {
    return on_gpu(w, at::kByte) && w.dim() == 2 && w.stride(1) == 1 && w.size(0) >= n && w.size(1) >= m;
}
bool whole(const at::Tensor &t, at::ScalarType dt) { return on_gpu(t, dt) && t.is_contiguous(); }

template <typename T>
T *ptr(const at::Tensor &t) { return static_cast<T *>(t.data_ptr()); }
const uint8_t *u8(const at::Tensor &t) { return ptr<const uint8_t>(t); }

// ---- torch.ops.rwkv.* ------------------------------------------------------------------------------------------------
template <typename... A>
void in_python(const char *name, A &&...args) {
    pybind11::gil_scoped_acquire gil;
    pybind11::module_::import("rwkvstic_amd.ops").attr(name)(std::forward<A>(args)...);
}

bool try_one(int64_t N, int64_t M, const at::Tensor &x, const at::Tensor &w, const at::Tensor &y, const at::Tensor &r) {
    const auto dt = x.scalar_type();
    const Stream st = current();
    if ((dt != at::kFloat && dt != at::kDouble) || !scratch_fits(st, x)) return false;
    if (!vec(x, dt) || !vec(y, dt) || !vec(r, dt) || !codes(w, N, M)) return false;
    if (N <= 0 || M <= 0 || x.numel() < N || r.numel() < N || y.numel() < M) return false;
    if (dt == at::kFloat) {
        const at::Tensor ws = bytes(lib.mm8_workspace_bytes(N, M, 1), x);
        check(lib.mm8_one(handle(st), N, M, ptr<float>(x), u8(w), w.stride(0), ptr<float>(y), ptr<float>(r), ws.data_ptr(), ws.numel()));
    } else {
        const at::Tensor ws = bytes(lib.mm8_f64_workspace_bytes(N, M, 1), x);
        check(lib.mm8_one_f64(handle(st), N, M, ptr<double>(x), u8(w), w.stride(0), ptr<double>(y), ptr<double>(r), ws.data_ptr(), ws.numel()));
    }
    return true;
}

void mm8_one(int64_t N, int64_t M, at::Tensor &x, at::Tensor &w, at::Tensor &y, at::Tensor &r) {
    if (!try_one(N, M, x, w, y, r)) in_python("mm8_one", N, M, x, w, y, r);
}

using T3 = const at::Tensor *const (&)[3];
bool try_three(int64_t N, int64_t M, T3 x, T3 w, T3 y, T3 r) {
    const auto dt = x[0]->scalar_type();
    const Stream st = current();
    if ((dt != at::kFloat && dt != at::kDouble) || N <= 0 || M <= 0 || !scratch_fits(st, *x[0])) return false;
    for (int i = 0; i < 3; ++i) {
        if (!vec(*x[i], dt) || !vec(*y[i], dt) || !vec(*r[i], dt) || !codes(*w[i], N, M)) return false;
        if (x[i]->numel() < N || r[i]->numel() < N || y[i]->numel() < M) return false;
    }
    auto call = [&](auto fn, auto bytes_fn, auto zero) {
        using T = decltype(zero);
        const at::Tensor ws = bytes(bytes_fn(N, M, 3), *x[0]);
        check(fn(handle(st), N, M, ptr<T>(*x[0]), ptr<T>(*x[1]), ptr<T>(*x[2]), u8(*w[0]), w[0]->stride(0), u8(*w[1]), w[1]->stride(0),
                 u8(*w[2]), w[2]->stride(0), ptr<T>(*y[0]), ptr<T>(*y[1]), ptr<T>(*y[2]), ptr<T>(*r[0]), ptr<T>(*r[1]), ptr<T>(*r[2]),
                 ws.data_ptr(), ws.numel()));
    };
    if (dt == at::kFloat) call(lib.mm8_three, lib.mm8_workspace_bytes, 0.f);
    else call(lib.mm8_three_f64, lib.mm8_f64_workspace_bytes, 0.0);
    return true;
}

void mm8_three(int64_t N, int64_t M, at::Tensor &x, at::Tensor &x1, at::Tensor &x2, at::Tensor &w, at::Tensor &w1, at::Tensor &w2,
               at::Tensor &y, at::Tensor &y1, at::Tensor &y2, at::Tensor &r, at::Tensor &r1, at::Tensor &r2) {
    const at::Tensor *const xs[3] = {&x, &x1, &x2}, *const ws[3] = {&w, &w1, &w2}, *const ys[3] = {&y, &y1, &y2}, *const rs[3] = {&r, &r1, &r2};
    if (!try_three(N, M, xs, ws, ys, rs)) in_python("mm8_three", N, M, x, x1, x2, w, w1, w2, y, y1, y2, r, r1, r2);
}

void wkv_forward(int64_t B, int64_t T, int64_t C, at::Tensor &w, at::Tensor &u, at::Tensor &k, at::Tensor &v, at::Tensor &y,
                 at::Tensor &aa, at::Tensor &bb, at::Tensor &pp) {
    bool ok = B > 0 && T > 0 && C > 0;
    for (const at::Tensor *t : {&w, &u, &k, &v, &y, &aa, &bb, &pp}) ok = ok && whole(*t, at::kDouble);
    for (const at::Tensor *t : {&k, &v, &y}) ok = ok && t->numel() / C / T >= B;
    for (const at::Tensor *t : {&aa, &bb, &pp}) ok = ok && t->numel() / C >= B;
    for (const at::Tensor *t : {&w, &u}) ok = ok && t->numel() >= C;
    if (!ok) return in_python("wkv_forward", B, T, C, w, u, k, v, y, aa, bb, pp);
    check(lib.wkv_forward_f64(handle(current()), B, T, C, ptr<double>(w), ptr<double>(u), ptr<double>(k), ptr<double>(v), ptr<double>(y),
                              ptr<double>(aa), ptr<double>(bb), ptr<double>(pp)));
}

void register_ops(const std::vector<std::string> &schemas) {
    static torch::Library *published = nullptr;      // (lives as long as the process: operators are looked up until its end)
    if (published) return;
    auto *l = new torch::Library(torch::Library::DEF, "rwkv", std::nullopt, __FILE__, __LINE__);
    for (const std::string &s : schemas) l->def(s.c_str());
    l->impl("wkv_forward", c10::DispatchKey::CUDA, TORCH_FN(wkv_forward));
    l->impl("mm8_one", c10::DispatchKey::CUDA, TORCH_FN(mm8_one));
    l->impl("mm8_three", c10::DispatchKey::CUDA, TORCH_FN(mm8_three));
    published = l;
}

// ---- stand-alone kernels: the result, or None where the Python function has to look at the call ------------------------
using Arg = pybind11::handle;

// The library's answer to a call from Python, made without the interpreter's lock: a launch waits where the queue is full.
// (The operators above come through torch's dispatcher, which has let go of it.)
template <typename F, typename... A>
void unlocked(F fn, A... args) {
    pybind11::gil_scoped_release gil;
    check(fn(handle(current()), args...));
}

const at::Tensor *tensor(Arg a) { return THPVariable_CheckExact(a.ptr()) ? &THPVariable_Unpack(a.ptr()) : nullptr; }

struct Product {
    const at::Tensor *x, *packed, *r_row, *m_row, *r_col = nullptr, *m_col = nullptr;
    at::Tensor y;
    const float *col(const at::Tensor *t) const { return t ? ptr<const float>(*t) : nullptr; }
};

bool product(Product &p, decltype(lib.packed_bytes) bytes_fn, Arg x, Arg packed, int64_t n_in, int64_t n_out, Arg r_row, Arg m_row,
             Arg r_col, Arg m_col, Arg out) {
    p.x = tensor(x); p.packed = tensor(packed); p.r_row = tensor(r_row); p.m_row = tensor(m_row);
    if (!p.x || !p.packed || !p.r_row || !p.m_row || n_in <= 0 || n_out <= 0) return false;
    if (!whole(*p.x, at::kFloat) || p.x->dim() != 2 || p.x->size(1) != n_in || !whole(*p.packed, at::kByte) ||
        !whole(*p.r_row, at::kFloat) || !whole(*p.m_row, at::kDouble)) return false;
    if (p.packed->numel() < (int64_t)bytes_fn(n_in, n_out) || p.r_row->numel() < n_in || p.m_row->numel() < n_in) return false;
    for (auto [h, t] : {std::pair{r_col, &p.r_col}, std::pair{m_col, &p.m_col}}) {
        if (h.is_none()) continue;
        *t = tensor(h);
        if (!*t || !whole(**t, at::kFloat) || (*t)->numel() < n_out) return false;
    }
    if (out.is_none()) p.y = at::empty({p.x->size(0), n_out}, p.x->options().dtype(at::kDouble));
    else {
        const at::Tensor *t = tensor(out);
        if (!t || !whole(*t, at::kDouble) || t->numel() < p.x->size(0) * n_out) return false;
        p.y = *t;
    }
    return true;
}

pybind11::object mm8_packed(Arg x, Arg packed, int64_t n_in, int64_t n_out, Arg r_row, Arg m_row, Arg r_col, Arg m_col, Arg out) {
    Product p;
    if (!product(p, lib.packed_bytes, x, packed, n_in, n_out, r_row, m_row, r_col, m_col, out)) return pybind11::none();
    unlocked(lib.mm8_packed, p.x->size(0), n_in, n_out, ptr<float>(*p.x), u8(*p.packed), ptr<float>(*p.r_row), ptr<double>(*p.m_row),
             p.col(p.r_col), p.col(p.m_col), ptr<double>(p.y));
    return out.is_none() ? pybind11::cast(p.y) : pybind11::reinterpret_borrow<pybind11::object>(out);
}

pybind11::object mm8_m16(Arg x, Arg packed, int64_t n_in, int64_t n_out, Arg r_row, Arg m_row, Arg r_col, Arg m_col, Arg out, Arg workspace) {
    Product p;
    if (!product(p, lib.packed_m16_bytes, x, packed, n_in, n_out, r_row, m_row, r_col, m_col, out)) return pybind11::none();
    const int64_t B = p.x->size(0);
    at::Tensor ws;
    if (workspace.is_none()) ws = bytes(lib.mm8_m16_workspace_bytes(B, n_in), *p.x);
    else if (const at::Tensor *t = tensor(workspace); t && t->is_cuda() && t->is_contiguous()) ws = *t;
    else return pybind11::none();
    unlocked(lib.mm8_m16, B, n_in, n_out, ptr<float>(*p.x), u8(*p.packed), ptr<float>(*p.r_row), ptr<double>(*p.m_row),
             p.col(p.r_col), p.col(p.m_col), ptr<double>(p.y), ws.data_ptr(), (size_t)ws.numel());
    return out.is_none() ? pybind11::cast(p.y) : pybind11::reinterpret_borrow<pybind11::object>(out);
}

pybind11::object wkv_f32(Arg w, Arg u, Arg k, Arg v, Arg aa, Arg bb, Arg pp) {
    const Arg args[7] = {w, u, k, v, aa, bb, pp};
    const at::Tensor *t[7];
    for (int i = 0; i < 7; ++i) {
        t[i] = tensor(args[i]);
        if (!t[i] || !whole(*t[i], at::kFloat)) return pybind11::none();
    }
    if (t[2]->dim() != 3 || t[3]->sizes() != t[2]->sizes()) return pybind11::none();
    const int64_t B = t[2]->size(0), T = t[2]->size(1), C = t[2]->size(2);
    for (int i : {4, 5, 6}) if (t[i]->numel() < B * C) return pybind11::none();
    for (int i : {0, 1}) if (t[i]->numel() < C) return pybind11::none();
    at::Tensor y = at::empty_like(*t[2]);
    unlocked(lib.wkv_f32, B, T, C, ptr<float>(*t[0]), ptr<float>(*t[1]), ptr<float>(*t[2]), ptr<float>(*t[3]), ptr<float>(y),
             ptr<float>(*t[4]), ptr<float>(*t[5]), ptr<float>(*t[6]));
    return pybind11::cast(y);
}

}  // namespace

PYBIND11_MODULE(_rwkv_torch, m) {
    m.def("bind", &bind);
    m.def("register_ops", &register_ops);
    m.def("mm8_packed", &mm8_packed);
    m.def("mm8_m16", &mm8_m16);
    m.def("wkv_f32", &wkv_f32);
}
