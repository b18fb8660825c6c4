// The host side of the operators as a Python extension module: argument checks, output allocation and the C-ABI call of each hot
// operator in one native call.  At decode sizes a launch takes the GPU 2 - 7 us, and the same steps in Python (a dozen tensor
// checks, torch.empty, the current stream, a ctypes call) took 10 - 22 us, so that a program that launches eagerly waited for
// its host; here they take 3 - 5 us.
//
// Every function takes its arguments by position (the Python modules of the package hold the signatures and their defaults) and
// raises what the checks of _lib.py raise: TypeError for something that is not a GPU tensor of the expected type, ValueError for
// a wrong shape or layout, RuntimeError for an error code of the C ABI.  The module keeps scratch buffers and tables per device
// (and stream); they are touched with the GIL held only.  It is released while memory is allocated and kernels are launched: either may
// wait for the GPU, and other threads of the program go on meanwhile.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <climits>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/qwen_tailor_hip.h"

namespace {

using at::Tensor;
using at::ScalarType;

constexpr ScalarType BF16 = at::kBFloat16, F32 = at::kFloat, I32 = at::kInt, F16 = at::kHalf, U8 = at::kByte;
constexpr int64_t HV = 16, DK = 128, DV = 128, CD = 6144, PW = 8224, QKV_W = 5120, ANY = -1;

struct Error {                              // a Python exception to be raised
    PyObject* type;
    std::string text;
};
struct Raised {};                           // ... that is already set
struct Ref {                                // an owned reference (a null one is an exception that is already set)
    PyObject* o;
    explicit Ref(PyObject* p) : o(p) {
        if (!o) throw Raised{};
    }
    Ref(const Ref&) = delete;
    ~Ref() { Py_DECREF(o); }
};
[[noreturn]] void type_error(const std::string& s) { throw Error{PyExc_TypeError, s}; }
[[noreturn]] void value_error(const std::string& s) { throw Error{PyExc_ValueError, s}; }

template <typename V>
std::string shape_text(const V& v) {        // as Python prints a tuple (None for a free entry)
    std::string r = "(";
    for (size_t i = 0; i < v.size(); i++) r += (i ? ", " : "") + (v[i] == ANY ? std::string("None") : std::to_string(v[i]));
    return r + (v.size() == 1 ? ",)" : ")");
}
const char* dtype_text(ScalarType t) {
    switch (t) {
        case BF16: return "torch.bfloat16";
        case F32: return "torch.float32";
        case I32: return "torch.int32";
        case F16: return "torch.float16";
        case U8: return "torch.uint8";
        case at::kDouble: return "torch.float64";
        case at::kLong: return "torch.int64";
        default: return at::toString(t);
    }
}

const Tensor& gpu_tensor(PyObject* o, const char* name) {
    if (!THPVariable_Check(o) || !THPVariable_Unpack(o).is_cuda()) type_error(std::string(name) + ": expected a tensor on the GPU");
    return THPVariable_Unpack(o);
}
void check_shape(const Tensor& t, const char* name, std::initializer_list<int64_t> shape) {
    const auto have = t.sizes();
    bool ok = have.size() == shape.size();
    size_t i = 0;
    for (int64_t s : shape) ok = ok && (s == ANY || have[i] == s), i++;
    if (!ok) value_error(std::string(name) + ": expected shape " + shape_text(std::vector<int64_t>(shape)) + ", got " + shape_text(have.vec()));
}
void check_layout(const Tensor& t, ScalarType dtype, const char* name) {
    if (t.scalar_type() != dtype)
        type_error(std::string(name) + ": expected " + dtype_text(dtype) + ", got " + dtype_text(t.scalar_type()));
    if (!t.is_contiguous()) value_error(std::string(name) + ": must be contiguous");
}
// a contiguous GPU tensor of `dtype` (and of `shape`, where given; ANY entries are free)
const Tensor& dev(PyObject* o, ScalarType dtype, const char* name) {
    const Tensor& t = gpu_tensor(o, name);
    check_layout(t, dtype, name);
    return t;
}
const Tensor& dev(PyObject* o, ScalarType dtype, const char* name, std::initializer_list<int64_t> shape) {
    const Tensor& t = dev(o, dtype, name);
    check_shape(t, name, shape);
    return t;
}
// per-head parameter vectors are consumed as float32: anything else is converted
Tensor f32(PyObject* o, const char* name, int64_t n) {
    Tensor t = gpu_tensor(o, name);
    if (t.scalar_type() != F32 || !t.is_contiguous()) t = t.to(F32).contiguous();
    check_shape(t, name, {n});
    return t;
}
const Tensor& flat_conv_w(PyObject* o) {
    const Tensor& w = dev(o, BF16, "conv_w");
    if (w.numel() != CD * 4) value_error("conv_w: expected " + std::to_string(CD * 4) + " elements, got " + std::to_string(w.numel()));
    return w;
}

long integer(PyObject* o) {                 // an int, or what stands for one (__index__): a float or a string does not
    const Ref i(PyNumber_Index(o));
    const long v = PyLong_AsLong(i.o);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
}
// a size, offset or stride of a copy: int(o), held at the ends of the range (no tensor is that large, so the range check refuses it)
long extent(PyObject* o) {
    int beyond = 0;
    long v;
    if (PyLong_CheckExact(o)) {
        v = PyLong_AsLongAndOverflow(o, &beyond);
    } else {
        const Ref i(PyNumber_Long(o));
        v = PyLong_AsLongAndOverflow(i.o, &beyond);
    }
    return beyond > 0 ? LONG_MAX : beyond < 0 ? LONG_MIN : v;
}
float real(PyObject* o) {                   // float(o)
    const Ref f(PyNumber_Float(o));
    return (float)PyFloat_AS_DOUBLE(f.o);
}
bool truth(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw Raised{};
    return v != 0;
}

struct Unlocked {                           // the GIL released; nothing of Python's may be touched meanwhile
    PyThreadState* state = PyEval_SaveThread();
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F>
auto unlocked(F f) {
    const Unlocked u;
    return f();
}

Tensor empty(at::IntArrayRef size, ScalarType dtype, const Tensor& like) {
    return Tensor(at::detail::empty_cuda(size, dtype, like.device(), std::nullopt));
}
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }
const char* code_text(int rc) {
    switch (rc) {
        case -1: return "bad dimension";
        case -2: return "misaligned pointer";
        case -3: return "null pointer";
        case -4: return "unsupported shape";
        case -5: return "kernel launch failed";
        case -6: return "workspace too small";
        case -7: return "size beyond the maximum of the allocation-free entry point";
        default: return "unknown error";
    }
}
void check(int rc, const char* name) {
    if (rc) throw Error{PyExc_RuntimeError, std::string(name) + " failed: " + code_text(rc)};
}
int dim32(int64_t v) { return v > INT_MAX ? INT_MAX : (int)v; }

PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }
PyObject* wrap(std::initializer_list<Tensor> ts) {
    PyObject* r = PyTuple_New(ts.size());
    Py_ssize_t i = 0;
    for (const Tensor& t : ts) PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(t));
    return r;
}

// ---- buffers that outlive a call ----------------------------------------------------------------------------------------
// Never destroyed: at interpreter exit the allocator that owns their memory may be gone already.  A buffer that is outgrown is
// kept: a HIP graph captured earlier replays with its address.
std::vector<Tensor>& retired() {
    static auto* v = new std::vector<Tensor>;
    return *v;
}
// Scratch memory for a kernel's partial results (the C ABI never allocates): one buffer per (purpose, device, stream), because
// launches on different streams may overlap.  `first`: size of the first allocation, so that growth is rare.  Under HIP graph capture
// it is memory of the graph, free for the next call once this one has been recorded: graphs captured on one stream may be replayed
// side by side, and beside eager calls.
// The launches of one call must follow each other on their stream: a call holds `busy` over them, so that another thread that uses the
// same stream (its buffer, then) does not come in between.  It is taken without the GIL.
struct Scratch {
    Tensor buf;
    std::mutex* busy;                       // null: the buffer is not shared
};
struct Busy {
    std::mutex* m;
    explicit Busy(std::mutex* busy) : m(busy) {
        if (m) m->lock();
    }
    Busy(const Busy&) = delete;
    ~Busy() {
        if (m) m->unlock();
    }
};
enum Purpose { ATTN_B, PREFILL_ATTENTION };
Scratch workspace(int purpose, const Tensor& like, long bytes, long first) {
    if (capturing()) return {unlocked([&] { return empty({bytes}, U8, like); }), nullptr};
    struct Kept {
        Tensor buf;
        std::mutex busy;
    };
    static auto* m = new std::map<std::tuple<int, int, void*>, Kept>;
    Kept& k = (*m)[{purpose, (int)like.device().index(), stream()}];
    if (!k.buf.defined() || k.buf.numel() < bytes) {
        Tensor larger = unlocked([&] { return empty({std::max(bytes, first)}, U8, like); });
        if (k.buf.defined()) retired().push_back(k.buf);         // (also one that another thread has made meanwhile)
        k.buf = larger;
    }
    return {k.buf, &k.busy};
}
constexpr long WS_FIRST = 32 << 20;         // attn_b: enough for 256 sequences x 4 rows

// A table of constants per device, written by a kernel on whichever stream asks first.  It is handed to other streams and kept only
// once it has been written: the first use waits for its stream (once per device, and when a table grows).  While a HIP graph is
// being captured nothing has run, and nothing may be waited for: the table then belongs to the graph, whose replays write it, and
// is not kept.  need: the rows that the caller asks for.
template <typename Build>
Tensor table(std::map<int, Tensor>& m, const Tensor& like, int64_t need, std::initializer_list<int64_t> shape, ScalarType dtype, Build build) {
    const int device = like.device().index();
    if (const auto it = m.find(device); it != m.end() && it->second.size(0) >= need) return it->second;
    Tensor t = unlocked([&] {
        Tensor n = empty(shape, dtype, like);
        build(n);
        if (!capturing()) c10::hip::getCurrentHIPStream().synchronize();
        return n;
    });
    if (capturing()) return t;
    Tensor& kept = m[device];
    if (kept.defined()) retired().push_back(kept);               // (also one that another thread has made meanwhile)
    return kept = t;
}
Tensor silu_table(const Tensor& like) {
    static auto* m = new std::map<int, Tensor>;
    return table(*m, like, 0, {qt_silu_table_bytes() / 2}, BF16,
                 [](const Tensor& t) { check(qt_silu_table_build(t.data_ptr(), stream()), "qt_silu_table_build"); });
}
// the (cos, sin) pairs of the rotary embedding for positions 0 .. n_pos - 1; grown in steps of 16384 positions
Tensor rope_table(const Tensor& like, int64_t n_pos) {
    static auto* m = new std::map<int, Tensor>;
    return table(*m, like, n_pos, {(std::max<int64_t>(n_pos, 1) + 16383) / 16384 * 16384, 32, 2}, F32,
                 [](const Tensor& t) { check(qt_rope_table_build(t.data_ptr(), dim32(t.size(0)), stream()), "qt_rope_table_build"); });
}

// ---- projections ----------------------------------------------------------------------------------------------------------
Tensor do_rms_rows(const Tensor& x, const Tensor& nw, float eps) {
    Tensor y = empty(x.sizes(), BF16, x);
    check(qt_rms_rows(x.data_ptr(), nw.data_ptr(), y.data_ptr(), dim32(x.size(0)), dim32(x.size(1)), eps, stream()), "qt_rms_rows");
    return y;
}
Tensor do_gated_norm(const Tensor& y, const Tensor& proj, const Tensor& gw, float eps) {
    Tensor out = empty({y.size(0), HV * DV}, BF16, y);
    check(qt_gated_rmsnorm(y.data_ptr(), proj.data_ptr(), gw.data_ptr<float>(), out.data_ptr(), y.size(0), eps, stream()), "qt_gated_rmsnorm");
    return out;
}

// rms_rows(x, nw, eps, f32)
PyObject* rms_rows(PyObject* const* a) {
    const Tensor& x = dev(a[0], BF16, "x", {ANY, ANY});
    const Tensor& nw = dev(a[1], BF16, "nw", {x.size(1)});
    const float eps = real(a[2]);
    const bool wide = truth(a[3]);
    return wrap(unlocked([&] {
        Tensor y = do_rms_rows(x, nw, eps);
        return wide ? y.to(F32) : y;
    }));
}

// fused_gemv(W, x, nw, eps, res, swiglu, gnorm)
PyObject* fused_gemv(PyObject* const* a) {
    if (PyTuple_Check(a[0]) || PyList_Check(a[0])) type_error("W: compressed weight pairs are not supported, pass the plain bf16 [N, K] matrix");
    const Tensor& W = dev(a[0], BF16, "W", {ANY, ANY});
    const int64_t N = W.size(0), K = W.size(1);
    const Tensor& xin = gpu_tensor(a[1], "x");
    if (xin.dim() < 1 || xin.size(-1) != K) value_error("x: last dimension must be " + std::to_string(K) + ", got " + shape_text(xin.sizes().vec()));
    const bool has_nw = a[2] != Py_None, has_res = a[4] != Py_None, swiglu = truth(a[5]), has_gnorm = a[6] != Py_None;
    Tensor x = xin;
    if (x.scalar_type() == F32) {
        if (has_nw || has_gnorm) value_error("float32 x carries already normalised values: no prologue may follow");
        x = x.to(BF16);                                          // exact: the values are bf16 values
    }
    if (x.dim() != 2) x = x.reshape({-1, K});
    check_layout(x, BF16, "x");
    const int64_t M = x.size(0);
    if (has_nw && has_gnorm) value_error("nw and gnorm are exclusive");
    if (swiglu && has_res) value_error("swiglu and res are exclusive");
    const float eps = has_nw || has_gnorm ? real(a[3]) : 0.f;    // (without a prologue nothing looks at it)
    Tensor proj, gw;
    if (has_gnorm) {
        const Ref pp(PySequence_GetItem(a[6], 0)), pg(PySequence_GetItem(a[6], 1));
        check_shape(x, "y", {ANY, HV * DV});
        proj = gpu_tensor(pp.o, "proj").reshape({M, PW});
        check_layout(proj, BF16, "proj");
        gw = f32(pg.o, "gw", DV);
    }
    const int epi = swiglu ? 2 : has_res ? 1 : 0;
    const int64_t n_out = swiglu ? N / 2 : N;
    Tensor res;
    if (has_res) {
        res = gpu_tensor(a[4], "res");
        if (res.dim() != 2 || res.size(1) != N) res = res.reshape({-1, N});
        check_layout(res, BF16, "res");
        check_shape(res, "res", {M, N});
    }
    const Tensor* nw = has_nw ? &dev(a[2], BF16, "nw", {K}) : nullptr;
    std::vector<int64_t> shape = xin.sizes().vec();
    shape.back() = n_out;
    return wrap(unlocked([&] {
        if (has_gnorm) x = do_gated_norm(x, proj, gw, eps);
        Tensor y = empty(shape, BF16, x);
        const void* rp = has_res ? res.data_ptr() : nullptr;
        if (has_nw) {
            // one launch for the shapes that have it, otherwise the prologue as its own kernel
            const int rc = qt_fused_gemv_rms(W.data_ptr(), x.data_ptr(), nw->data_ptr(), eps, rp, y.data_ptr(), dim32(M), dim32(N), dim32(K), epi, stream());
            if (rc == 0) return y;
            if (rc != -4) check(rc, "qt_fused_gemv_rms");
            x = do_rms_rows(x, *nw, eps);
        }
        check(qt_fused_gemv(W.data_ptr(), x.data_ptr(), rp, y.data_ptr(), dim32(M), dim32(N), dim32(K), epi, stream()), "qt_fused_gemv");
        return y;
    }));
}

// gated_norm(y [rows, 2048], proj, gw, eps)
PyObject* gated_norm(PyObject* const* a) {
    const Tensor& y = dev(a[0], BF16, "y", {ANY, HV * DV});
    const Tensor &proj = dev(a[1], BF16, "proj", {y.size(0), PW}), gw = f32(a[2], "gw", DV);
    const float eps = real(a[3]);
    return wrap(unlocked([&] { return do_gated_norm(y, proj, gw, eps); }));
}

// ---- recurrent steps ------------------------------------------------------------------------------------------------------
struct Step {                               // the operands of a decode step
    const Tensor &proj, &ssm, &conv, &slots, &pos, &w;
    Tensor A, dtb;
    int B, n_slots;
};
// (proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, slots, pos)
Step step_operands(PyObject* const* a) {
    const Tensor& proj = dev(a[0], BF16, "proj", {ANY, PW});
    const int64_t B = proj.size(0);
    const Tensor& ssm = dev(a[5], F32, "ssm_pool", {ANY, HV, DV, DK});
    const int64_t n_slots = ssm.size(0);
    const Tensor& conv = dev(a[1], BF16, "conv_pool", {n_slots * 2, 3, CD});
    const Tensor &slots = dev(a[6], I32, "slots", {B}), &pos = dev(a[7], I32, "pos", {B}), &w = flat_conv_w(a[2]);
    return {proj, ssm, conv, slots, pos, w, f32(a[3], "A_log", HV), f32(a[4], "dt_bias", HV), dim32(B), dim32(n_slots)};
}
// decode_step(proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, slots, pos, rows_per_wg)
PyObject* decode_step(PyObject* const* a) {
    const Step s = step_operands(a);
    const int rows_per_wg = (int)integer(a[8]);
    return wrap(unlocked([&] {
        Tensor y = empty({s.proj.size(0), HV * DV}, BF16, s.proj);
        check(qt_gdn_decode_step(s.proj.data_ptr(), s.conv.data_ptr(), s.w.data_ptr(), s.A.data_ptr<float>(), s.dtb.data_ptr<float>(),
                                 s.ssm.data_ptr<float>(), s.slots.data_ptr<int>(), s.pos.data_ptr<int>(), y.data_ptr(), s.B, s.n_slots, rows_per_wg,
                                 stream()), "qt_gdn_decode_step");
        return y;
    }));
}
// decode_step_gnorm(proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, slots, pos, gw, eps)
PyObject* decode_step_gnorm(PyObject* const* a) {
    const Step s = step_operands(a);
    const Tensor gw = f32(a[8], "gw", DV);
    const float eps = real(a[9]);
    return wrap(unlocked([&] {
        Tensor out = empty({s.proj.size(0), HV * DV}, BF16, s.proj);
        check(qt_gdn_decode_step_gnorm(s.proj.data_ptr(), s.conv.data_ptr(), s.w.data_ptr(), s.A.data_ptr<float>(), s.dtb.data_ptr<float>(),
                                       s.ssm.data_ptr<float>(), s.slots.data_ptr<int>(), s.pos.data_ptr<int>(), gw.data_ptr<float>(), eps,
                                       out.data_ptr(), s.B, s.n_slots, stream()), "qt_gdn_decode_step_gnorm");
        return out;
    }));
}

// verify_step(proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, sslots, sels, pars, M, rows_per_wg)
PyObject* verify_step(PyObject* const* a) {
    const Tensor& ss = dev(a[6], I32, "sslots");
    if (ss.dim() < 1) value_error("sslots: expected one entry per sequence");
    const int64_t B = ss.size(0), M = integer(a[9]);
    const Tensor& proj = dev(a[0], BF16, "proj", {B * M, PW});
    const Tensor& ssm = dev(a[5], F32, "ssm_pool", {ANY, M, HV, DV, DK});
    const int64_t n = ssm.size(0);
    const Tensor& conv = dev(a[1], BF16, "conv_pool", {n * 2, M, 3, CD});
    const Tensor &sels = dev(a[7], I32, "sels", {B}), &pars = dev(a[8], I32, "pars", {B}), &w = flat_conv_w(a[2]);
    const Tensor A = f32(a[3], "A_log", HV), dtb = f32(a[4], "dt_bias", HV);
    const int rows_per_wg = (int)integer(a[10]);
    return wrap(unlocked([&] {
        Tensor y = empty({B * M, HV * DV}, BF16, proj);
        check(qt_gdn_verify_step(proj.data_ptr(), conv.data_ptr(), w.data_ptr(), A.data_ptr<float>(), dtb.data_ptr<float>(), ssm.data_ptr<float>(),
                                 ss.data_ptr<int>(), sels.data_ptr<int>(), pars.data_ptr<int>(), y.data_ptr(), dim32(B), dim32(M), dim32(n),
                                 rows_per_wg, stream()), "qt_gdn_verify_step");
        return y;
    }));
}

// deltanet(proj, conv_snap, conv_w, A_log, dt_bias, ssm_snap, sel, rows_per_wg)
PyObject* deltanet(PyObject* const* a) {
    const Tensor& proj = dev(a[0], BF16, "proj", {ANY, PW});
    const int64_t M = proj.size(0);
    const Tensor &conv = dev(a[1], BF16, "conv_snap", {ANY, 3, CD}), &ssm = dev(a[5], F32, "ssm_snap", {ANY, HV, DV, DK});
    const int64_t S = ssm.size(0);
    if (conv.size(0) != S) value_error("conv_snap and ssm_snap must hold the same number of snapshots");
    const Tensor &sel = dev(a[6], I32, "sel", {1}), &w = flat_conv_w(a[2]);
    const Tensor A = f32(a[3], "A_log", HV), dtb = f32(a[4], "dt_bias", HV);
    const int rows_per_wg = (int)integer(a[7]);
    Tensor y, cs, st;
    unlocked([&] {
        y = empty({M, HV * DV}, BF16, proj), cs = empty({M, 3, CD}, BF16, proj), st = empty({M, HV, DV, DK}, F32, proj);
        check(qt_gdn_deltanet(proj.data_ptr(), conv.data_ptr(), w.data_ptr(), A.data_ptr<float>(), dtb.data_ptr<float>(), ssm.data_ptr<float>(),
                              sel.data_ptr<int>(), y.data_ptr(), cs.data_ptr(), st.data_ptr<float>(), dim32(M), dim32(S), rows_per_wg, stream()),
              "qt_gdn_deltanet");
    });
    return wrap({y, cs, st});
}

// ---- decode / verify attention --------------------------------------------------------------------------------------------
struct Pool {
    const Tensor &K, &V, &slots, &pos;
    int64_t n_slots, Lmax;
};
Pool kv_pool(PyObject* kp, PyObject* vp, PyObject* slots, PyObject* pos, int64_t B) {
    const Tensor& K = dev(kp, BF16, "Kp", {ANY, 2, ANY, 256});
    const Tensor& V = dev(vp, BF16, "Vp", {K.size(0), K.size(1), K.size(2), K.size(3)});
    return {K, V, dev(slots, I32, "slots", {B}), dev(pos, I32, "pos", {B}), K.size(0), K.size(2)};
}
Scratch attn_scratch(PyObject* given, const Tensor& like, int64_t B, int64_t M, int64_t Lmax, long CH, const char* who) {
    const long bytes = qt_gqa_attn_workspace_bytes(dim32(B), dim32(M), dim32(Lmax), (int)CH);
    if (bytes < 0) value_error(std::string(who) + ": bad split size");
    if (given == Py_None) return workspace(ATTN_B, like, bytes, WS_FIRST);
    const Tensor& ws = dev(given, U8, "workspace");
    if (ws.numel() < bytes)
        value_error(std::string(who) + ": workspace of " + std::to_string(ws.numel()) + " bytes, " + std::to_string(bytes) + " needed");
    return {ws, nullptr};
}
int64_t sequences(int64_t R, int64_t M, const char* who, const char* limit) {
    if (M < 1 || M > 16 || R % M)
        value_error(std::string(who) + ": M = " + std::to_string(M) + " (" + limit + ") must divide the number of rows (" + std::to_string(R) + ")");
    return R / M;
}

// attn_b(q, k, v, Kp, Vp, slots, pos, M, split, workspace or None)
PyObject* attn_b(PyObject* const* a) {
    const Tensor& q = dev(a[0], BF16, "q", {ANY, 8, 256});
    const int64_t R = q.size(0), M = integer(a[7]), B = sequences(R, M, "attn_b", "1..16, as deltanet_bm");
    const Tensor &k = dev(a[1], BF16, "k", {R, 2, 256}), &v = dev(a[2], BF16, "v", {R, 2, 256});
    const Pool p = kv_pool(a[3], a[4], a[5], a[6], B);
    const long CH = integer(a[8]);
    const Scratch ws = attn_scratch(a[9], q, B, M, p.Lmax, CH, "attn_b");
    return wrap(unlocked([&] {
        Tensor o = empty({R, 8, 256}, BF16, q);
        const Busy busy(ws.busy);
        check(qt_gqa_attn_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), p.K.data_ptr(), p.V.data_ptr(), p.slots.data_ptr<int>(), p.pos.data_ptr<int>(),
                                 o.data_ptr(), ws.buf.data_ptr(), ws.buf.numel(), dim32(B), dim32(M), dim32(p.Lmax), dim32(p.n_slots), (int)CH, stream()),
              "qt_gqa_attn_decode");
        return o;
    }));
}

// attn_layer_b(qkv, q_norm, k_norm, Kp, Vp, slots, pos, M, eps, split, workspace or None)
PyObject* attn_layer_b(PyObject* const* a) {
    const Tensor& qkv = dev(a[0], BF16, "qkv", {ANY, QKV_W});
    const int64_t R = qkv.size(0), M = integer(a[7]), B = sequences(R, M, "attn_layer_b", "1..16");
    const Tensor &qn = dev(a[1], BF16, "q_norm", {256}), &kn = dev(a[2], BF16, "k_norm", {256});
    const Pool p = kv_pool(a[3], a[4], a[5], a[6], B);
    const long CH = integer(a[9]);
    const Scratch ws = attn_scratch(a[10], qkv, B, M, p.Lmax, CH, "attn_layer_b");
    const Tensor table = rope_table(qkv, p.Lmax);
    const float eps = real(a[8]);
    return wrap(unlocked([&] {
        Tensor out = empty({R, 2048}, BF16, qkv);
        const Busy busy(ws.busy);
        check(qt_gqa_attn_layer_decode(qkv.data_ptr(), qn.data_ptr(), kn.data_ptr(), table.data_ptr(), dim32(table.size(0)), p.K.data_ptr(), p.V.data_ptr(),
                                       p.slots.data_ptr<int>(), p.pos.data_ptr<int>(), out.data_ptr(), ws.buf.data_ptr(), ws.buf.numel(), dim32(B), dim32(M),
                                       dim32(p.Lmax), dim32(p.n_slots), (int)CH, eps, stream()), "qt_gqa_attn_layer_decode");
        return out;
    }));
}

// ---- prefill attention ----------------------------------------------------------------------------------------------------
// sdpa(q, k, v): the checks that need no arithmetic on floats; causal, scale 256^-0.5
PyObject* sdpa(PyObject* const* a) {
    const auto& qin = THPVariable_Check(a[0]) ? THPVariable_Unpack(a[0]) : Tensor();
    if (!qin.defined() || qin.dim() != 4 || qin.size(0) != 1 || qin.size(1) != 8 || qin.size(3) != 256 || qin.scalar_type() != BF16 || !qin.is_cuda())
        value_error("q: expected [1, 8, S, 256] bf16 on the GPU" + (qin.defined() ? ", got " + shape_text(qin.sizes().vec()) + " " + dtype_text(qin.scalar_type()) : std::string()));
    Tensor q = qin;
    const int64_t S = q.size(2);
    for (int i = 1; i < 3; i++) {
        const std::string name = i == 1 ? "k" : "v";
        if (!THPVariable_Check(a[i])) value_error(name + ": expected [1, 2, L, 256] bf16 on the GPU");
        const Tensor& t = THPVariable_Unpack(a[i]);
        if (t.dim() != 4 || t.size(0) != 1 || t.size(1) != 2 || t.size(3) != 256 || t.scalar_type() != BF16 || !t.is_cuda())
            value_error(name + ": expected [1, 2, L, 256] bf16 on the GPU");
        if (t.stride(3) != 1 || t.stride(2) != 256) value_error(name + ": rows must be contiguous");
    }
    const Tensor &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
    if (k.sizes() != v.sizes() || k.stride(1) != v.stride(1)) value_error("k and v must have the same shape and head stride");
    const int64_t L = k.size(2);
    if (L < S) value_error("fewer keys than queries");
    const bool token_major = S > 1 && q.stride(1) == 256 && q.stride(2) == 2048 && q.stride(3) == 1 && !((uintptr_t)q.data_ptr() & 15);
    // launches that would leave half of the CUs idle are split along the keys; their parts meet in a workspace
    const long bytes = qt_gqa_prefill_workspace_bytes_for(dim32(S), dim32(L), dim32(L - S));
    const Scratch ws = bytes > 0 ? workspace(PREFILL_ATTENTION, q, bytes, 0) : Scratch{Tensor(), nullptr};
    return wrap(unlocked([&] {
        Tensor out;
        if (token_major) {
            out = empty({1, S, 8, 256}, BF16, q).transpose(1, 2);    // a transposed view of token-major rows: neither side is copied
        } else {
            q = q.contiguous();
            out = empty(q.sizes(), BF16, q);
        }
        const Busy busy(ws.busy);
        check(qt_gqa_prefill_causal_strided(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), bytes > 0 ? ws.buf.data_ptr() : nullptr,
                                            std::max(bytes, 0L), dim32(S), dim32(L), dim32(L - S), token_major ? 256 : S * 256, token_major ? 2048 : 256,
                                            k.stride(1), stream()), "qt_gqa_prefill_causal");
        return out;
    }));
}

// qkv_prep(qkv, q_norm, k_norm, pos, M, eps, max_pos or None)
PyObject* qkv_prep(PyObject* const* a) {
    const Tensor& qkv = dev(a[0], BF16, "qkv", {ANY, QKV_W});
    const int64_t R = qkv.size(0), M = integer(a[4]);
    if (M < 1 || R % M) value_error("qkv_prep: M = " + std::to_string(M) + " must divide the number of rows (" + std::to_string(R) + ")");
    const Tensor &pos = dev(a[3], I32, "pos", {R / M}), &qn = dev(a[1], BF16, "q_norm", {256}), &kn = dev(a[2], BF16, "k_norm", {256});
    const float eps = real(a[5]);
    const Tensor table = a[6] != Py_None ? rope_table(qkv, std::min(extent(a[6]), 1L << 40) + 1) : Tensor();
    Tensor q, k, v;
    unlocked([&] {
        q = empty({R, 8, 256}, BF16, qkv), k = empty({R, 2, 256}, BF16, qkv), v = empty({R, 2, 256}, BF16, qkv);
        check(qt_attn_qkv_prep_table(qkv.data_ptr(), qn.data_ptr(), kn.data_ptr(), pos.data_ptr<int>(), table.defined() ? table.data_ptr() : nullptr,
                                     table.defined() ? dim32(table.size(0)) : 0, q.data_ptr(), k.data_ptr(), v.data_ptr(), R, dim32(M), eps, stream()),
              "qt_attn_qkv_prep");
    });
    return wrap({q, k, v});
}

// out_gate(o, qkv)
PyObject* out_gate(PyObject* const* a) {
    const Tensor& qkv = dev(a[1], BF16, "qkv", {ANY, QKV_W});
    const int64_t R = qkv.size(0);
    const Tensor& o = dev(a[0], BF16, "o", {R, 8, 256});
    return wrap(unlocked([&] {
        Tensor out = empty({R, 2048}, BF16, qkv);
        check(qt_attn_out_gate(o.data_ptr(), qkv.data_ptr(), out.data_ptr(), R, stream()), "qt_attn_out_gate");
        return out;
    }));
}

// ---- chunked prefill ------------------------------------------------------------------------------------------------------
// conv_prep(proj, conv_state, conv_w)
PyObject* conv_prep(PyObject* const* a) {
    const Tensor& proj = dev(a[0], BF16, "proj", {ANY, PW});
    const int64_t S = proj.size(0);
    const Tensor &cs = dev(a[1], BF16, "conv_state", {3, CD}), &w = flat_conv_w(a[2]);
    const Tensor silu = silu_table(proj);
    Tensor q, k, v;
    unlocked([&] {
        q = empty({S, HV, DK}, BF16, proj), k = empty({S, HV, DK}, BF16, proj), v = empty({S, HV, DK}, BF16, proj);
        check(qt_gdn_conv_prep(proj.data_ptr(), cs.data_ptr(), w.data_ptr(), silu.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), dim32(S), stream()),
              "qt_gdn_conv_prep");
    });
    return wrap({q, k, v});
}

struct Records {
    Tensor ops, U, gC;
};
Records new_records(const Tensor& proj) {
    const int S = dim32(proj.size(0));
    return {empty({qt_gdn_chunk_ops_bytes(S) / 2}, F16, proj), empty({qt_gdn_chunk_u_bytes(S) / 2}, F16, proj), empty({qt_gdn_chunk_gc_bytes(S) / 4}, F32, proj)};
}
void phase_a_conv(const Tensor& proj, const Tensor& cs, const Tensor& w, const Tensor& silu, const Tensor& A, const Tensor& dtb, const Tensor* qkv,
                  void* conv_out, const Records& r) {
    check(qt_gdn_phase_a_conv(proj.data_ptr(), cs.data_ptr(), w.data_ptr(), silu.data_ptr(), A.data_ptr<float>(), dtb.data_ptr<float>(),
                              qkv ? qkv[0].data_ptr() : nullptr, qkv ? qkv[1].data_ptr() : nullptr, qkv ? qkv[2].data_ptr() : nullptr, conv_out,
                              r.ops.data_ptr(), r.U.data_ptr(), r.gC.data_ptr<float>(), dim32(proj.size(0)), stream()), "qt_gdn_phase_a_conv");
}

// phase_a(proj, conv_state, conv_w, A_log, dt_bias, (q, k, v) or None, want_qkv, conv_out or None) -> (q, k, v, ops, U, gC)
PyObject* phase_a(PyObject* const* a) {
    const Tensor& proj = dev(a[0], BF16, "proj", {ANY, PW});
    const int64_t S = proj.size(0);
    const Tensor A = f32(a[3], "A_log", HV), dtb = f32(a[4], "dt_bias", HV);
    Records r;
    if (a[5] != Py_None) {
        PyObject* seq = PySequence_Fast(a[5], "qkv: expected (q, k, v)");
        if (!seq) throw Raised{};
        static const char* names[3] = {"q", "k", "v"};
        Tensor t[3];
        try {
            if (PySequence_Fast_GET_SIZE(seq) != 3) value_error("qkv: expected (q, k, v)");
            for (int i = 0; i < 3; i++) t[i] = dev(PySequence_Fast_GET_ITEM(seq, i), BF16, names[i], {S, HV, DK});
        } catch (...) {
            Py_DECREF(seq);
            throw;
        }
        Py_DECREF(seq);
        unlocked([&] {
            r = new_records(proj);
            check(qt_gdn_phase_a(proj.data_ptr(), t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), A.data_ptr<float>(), dtb.data_ptr<float>(),
                                 r.ops.data_ptr(), r.U.data_ptr(), r.gC.data_ptr<float>(), dim32(S), stream()), "qt_gdn_phase_a");
        });
        return wrap({t[0], t[1], t[2], r.ops, r.U, r.gC});
    }
    const Tensor &cs = dev(a[1], BF16, "conv_state", {3, CD}), &w = flat_conv_w(a[2]);
    Tensor qkv[3];
    const bool want = truth(a[6]);
    void* conv_out = a[7] != Py_None ? dev(a[7], BF16, "conv_out", {3, CD}).data_ptr() : nullptr;
    const Tensor silu = silu_table(proj);
    unlocked([&] {
        r = new_records(proj);
        if (want)
            for (Tensor& t : qkv) t = empty({S, HV, DK}, BF16, proj);
        phase_a_conv(proj, cs, w, silu, A, dtb, want ? qkv : nullptr, conv_out, r);
    });
    PyObject* out = PyTuple_New(6);
    for (int i = 0; i < 3; i++) PyTuple_SET_ITEM(out, i, want ? wrap(qkv[i]) : (Py_INCREF(Py_None), Py_None));
    PyTuple_SET_ITEM(out, 3, wrap(r.ops));
    PyTuple_SET_ITEM(out, 4, wrap(r.U));
    PyTuple_SET_ITEM(out, 5, wrap(r.gC));
    return out;
}

// The buffer between phase B's chain and output workgroups and the host words its failures are reported in, per (device,
// stream).  gdn_nax makes them (it owns the caches that a caller can look at): snap_provider(device index, bytes) -> (buffer,
// pinned int32 tensor); words_provider(device index) -> the words alone; failed(device index) raises what the words say and
// resets them.
PyObject *snap_provider = nullptr, *words_provider = nullptr, *snap_failed = nullptr;
struct Snap {
    Tensor buf, words;
    std::mutex* busy;                                            // see Scratch
};
Snap snap_buffer(const Tensor& like, int64_t S) {
    const long bytes = qt_gdn_chunk_snap_bytes(dim32(S));
    const int device = like.device().index();
    if (!snap_provider) throw Error{PyExc_RuntimeError, "gdn_nax is not imported"};
    if (capturing()) {                                           // memory of the graph, see workspace(); its replays clear the flag area
        const Ref words(PyObject_CallFunction(words_provider, "i", device));
        return {unlocked([&] {
                    Tensor buf = empty({bytes / 2}, F16, like);
                    if (const long flags = qt_gdn_chunk_flag_bytes(dim32(S))) buf.narrow(0, 0, flags / 2).zero_();
                    return buf;
                }), THPVariable_Unpack(words.o), nullptr};
    }
    struct Kept {
        Tensor buf, words;
        std::mutex busy;
    };
    static auto* m = new std::map<std::pair<int, void*>, Kept>;
    Kept& k = (*m)[{device, stream()}];
    if (!k.buf.defined() || k.buf.numel() * 2 < bytes) {
        const Ref r(PyObject_CallFunction(snap_provider, "il", device, bytes));
        k.buf = THPVariable_Unpack(PyTuple_GET_ITEM(r.o, 0)), k.words = THPVariable_Unpack(PyTuple_GET_ITEM(r.o, 1));
    }
    const Snap s{k.buf, k.words, &k.busy};
    const int* w = s.words.data_ptr<int>();
    if (w[0] | w[1]) const Ref r(PyObject_CallFunction(snap_failed, "i", device));      // an earlier launch with these words has failed
    return s;
}
// set_hooks(snap_provider, words_provider, failed)
PyObject* set_hooks(PyObject* const* a) {
    for (int i = 0; i < 3; i++) Py_INCREF(a[i]);
    Py_XSETREF(snap_provider, a[0]);
    Py_XSETREF(words_provider, a[1]);
    Py_XSETREF(snap_failed, a[2]);
    Py_RETURN_NONE;
}
void phase_b_launch(const Records& r, const Snap& s, const Tensor& st, const Tensor& st_out, const Tensor* proj, const Tensor* gw, float eps,
                    const Tensor& out, int64_t S) {
    const Busy busy(s.busy);
    check(qt_gdn_phase_b_report(r.ops.data_ptr(), r.U.data_ptr(), r.gC.data_ptr<float>(), s.buf.data_ptr(), st.data_ptr<float>(), st_out.data_ptr<float>(),
                                proj ? proj->data_ptr() : nullptr, gw ? gw->data_ptr<float>() : nullptr, eps, out.data_ptr(), dim32(S),
                                s.words.data_ptr<int>(), stream()), "qt_gdn_phase_b");
}

Records given_records(PyObject* const* a, int S) {              // (ops, U, gC), of at least S tokens
    const Records r{dev(a[0], F16, "Tb"), dev(a[1], F16, "Am"), dev(a[2], F32, "gv")};
    if (r.ops.numel() * 2 < qt_gdn_chunk_ops_bytes(S) || r.U.numel() * 2 < qt_gdn_chunk_u_bytes(S) || r.gC.numel() * 4 < qt_gdn_chunk_gc_bytes(S))
        value_error("phase_b: the phase A records are too small for this many tokens");
    return r;
}
// phase_b(S, ops, U, gC, state)
PyObject* phase_b(PyObject* const* a) {
    const int64_t S = integer(a[0]);
    const Records r = given_records(a + 1, dim32(S));
    const Tensor state = dev(a[4], F32, "state").reshape({1, HV, DV, DK});
    const Snap s = snap_buffer(state, S);
    Tensor st_out, out;
    unlocked([&] {
        st_out = empty({1, HV, DV, DK}, F32, state), out = empty({S, HV, DV}, BF16, state);
        phase_b_launch(r, s, state, st_out, nullptr, nullptr, 0.f, out, S);
    });
    return wrap({out, st_out});
}
// phase_b_norm(proj, ops, U, gC, state, gw, eps): the gated norm follows in the same pass
PyObject* phase_b_norm(PyObject* const* a) {
    const Tensor& proj = dev(a[0], BF16, "proj", {ANY, PW});
    const int64_t S = proj.size(0);
    const Records r = given_records(a + 1, dim32(S));
    const Tensor state = dev(a[4], F32, "state").reshape({1, HV, DV, DK}), gw = f32(a[5], "gw", DV);
    const float eps = real(a[6]);
    const Snap s = snap_buffer(state, S);
    Tensor st_out, out;
    unlocked([&] {
        st_out = empty({1, HV, DV, DK}, F32, state), out = empty({S, HV * DV}, BF16, state);
        phase_b_launch(r, s, state, st_out, &proj, &gw, eps, out, S);
    });
    return wrap({out, st_out});
}

// gdn_core(proj, conv_state, ssm_state, conv_w, A_log, dt_bias, gw): both phases with the gated norm
PyObject* gdn_core(PyObject* const* a) {
    const Tensor& proj = dev(a[0], BF16, "proj", {ANY, PW});
    const int64_t S = proj.size(0);
    const Tensor cs = gpu_tensor(a[1], "conv_state").reshape({3, CD});
    check_layout(cs, BF16, "conv_state");
    const Tensor& w = flat_conv_w(a[3]);
    const Tensor A = f32(a[4], "A_log", HV), dtb = f32(a[5], "dt_bias", HV), gw = f32(a[6], "gw", DV);
    const Tensor state = dev(a[2], F32, "state").reshape({1, HV, DV, DK});
    const Snap s = snap_buffer(proj, S);
    const Tensor silu = silu_table(proj);
    Tensor conv_out, st_out, out;
    unlocked([&] {
        conv_out = empty({1, 3, CD}, BF16, proj), st_out = empty({1, HV, DV, DK}, F32, proj), out = empty({S, HV * DV}, BF16, proj);
        // a prompt of one chunk: one launch
        const int rc = qt_gdn_prefill_one(proj.data_ptr(), cs.data_ptr(), w.data_ptr(), silu.data_ptr(), A.data_ptr<float>(), dtb.data_ptr<float>(),
                                          conv_out.data_ptr(), s.buf.data_ptr(), state.data_ptr<float>(), st_out.data_ptr<float>(),
                                          gw.data_ptr<float>(), 1e-6f, out.data_ptr(), dim32(S), s.words.data_ptr<int>(), stream());
        if (rc != -4) return check(rc, "qt_gdn_prefill_one");
        const Records r = new_records(proj);
        phase_a_conv(proj, cs, w, silu, A, dtb, nullptr, conv_out.data_ptr(), r);
        phase_b_launch(r, s, state, st_out, &proj, &gw, 1e-6f, out, S);
    });
    return wrap({out, conv_out, st_out});
}

// ---- copies ---------------------------------------------------------------------------------------------------------------
struct Jobs {
    std::vector<PyObject*> held;                                 // (the caller's lists may change while the GIL is released)
    std::vector<void*> dst;
    std::vector<const void*> src;
    std::vector<long> meta;
    Jobs() = default;
    Jobs(const Jobs&) = delete;
    ~Jobs() {
        for (PyObject* o : held) Py_DECREF(o);
    }
    void reserve(size_t n) { held.reserve(2 * n), dst.reserve(n), src.reserve(n), meta.reserve(7 * n); }
    void add(PyObject* dest, PyObject* source, long n, long d0, long s0, long ny, long ds, long ss) {
        add(gpu_tensor(dest, "dst"), source, n, d0, s0, ny, ds, ss);
        Py_INCREF(dest);
        held.push_back(dest);
    }
    // (a destination that the caller keeps)
    void add(const Tensor& d, PyObject* source, long n, long d0, long s0, long ny, long ds, long ss) {
        add(d, gpu_tensor(source, "src"), n, d0, s0, ny, ds, ss);
        Py_INCREF(source);
        held.push_back(source);
    }
    void add(const Tensor& d, const Tensor& s, long n, long d0, long s0, long ny, long ds, long ss) {
        const auto who = [&] { return "blit_batch: job " + std::to_string(dst.size()); };
        if (d.scalar_type() != s.scalar_type() || (d.scalar_type() != BF16 && d.scalar_type() != F32))
            type_error(who() + ": bf16 or float32 tensors of one dtype expected");
        check_layout(d, d.scalar_type(), "dst");
        check_layout(s, s.scalar_type(), "src");
        if (n < 0 || ny < 0 || d0 < 0 || s0 < 0 || ds < 0 || ss < 0) value_error(who() + ": negative size, offset or stride");
        // `ny` rows of n elements from `first` on, `stride` apart, end inside t.  By subtraction and division: the sum
        // first + (ny - 1) * stride + n of sizes that no tensor has can pass 2^63
        auto fits = [n, ny](const Tensor& t, long first, long stride) {
            const long numel = t.numel();
            return n <= numel && first <= numel - n && (stride == 0 || ny - 1 <= (numel - n - first) / stride);
        };
        if (n && ny && !(fits(d, d0, ds) && fits(s, s0, ss))) value_error(who() + ": the copy leaves the source or the destination");
        dst.push_back(d.data_ptr());
        src.push_back(s.data_ptr());
        for (long v : {(long)d.element_size(), n, d0, s0, ny, ds, ss}) meta.push_back(v);
    }
    void add_zeros(const Tensor& d, long n, long d0, long ny, long ds) {   // `ny` rows of `n` zeros
        add(d, d, n, d0, d0, ny, ds, ds);                        // (the checks of the destination range)
        src.back() = nullptr;
        fills = true;
    }
    void add_zeros(PyObject* d, long n, long d0, long ny, long ds) {
        add_zeros(gpu_tensor(d, "dst"), n, d0, ny, ds);
        Py_INCREF(d);
        held.push_back(d);
    }
    bool fills = false;
    void run() const {
        if (dst.empty()) return;
        const int rc = unlocked([&] { return (fills ? qt_blit_fill_batch : qt_blit_batch)(dst.data(), src.data(), meta.data(), (int)dst.size(), stream()); });
        if (rc == -2) value_error("blit_batch: every copy must be 16-byte granular (base pointers, sizes, offsets, strides)");
        check(rc, "qt_blit_batch");
    }
};
struct Items {                                                   // the items of a list or tuple
    PyObject* seq;
    explicit Items(PyObject* o) : seq(PySequence_Fast(o, "expected a sequence")) {
        if (!seq) throw Raised{};
    }
    ~Items() { Py_DECREF(seq); }
    Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(seq); }
    PyObject* operator[](Py_ssize_t i) const {
        if (i < 0 || i >= size()) throw Error{PyExc_IndexError, "list index out of range"};
        return PySequence_Fast_GET_ITEM(seq, i);
    }
};

// blit_batch(jobs, zeros): sequences of (dst, src, n, d0, s0, ny, dstride, sstride) and of (dst, n, d0, ny, dstride)
PyObject* blit_batch(PyObject* const* a) {
    const Items jobs(a[0]), zeros(a[1]);
    Jobs j;
    j.reserve(jobs.size() + zeros.size());
    for (Py_ssize_t i = 0; i < jobs.size(); i++) {
        const Items t(jobs[i]);
        if (t.size() != 8) value_error("blit_batch: job " + std::to_string(i) + ": expected eight values");
        j.add(t[0], t[1], extent(t[2]), extent(t[3]), extent(t[4]), extent(t[5]), extent(t[6]), extent(t[7]));
    }
    for (Py_ssize_t i = 0; i < zeros.size(); i++) {
        const Items t(zeros[i]);
        if (t.size() != 5) value_error("blit_batch: zeros " + std::to_string(i) + ": expected five values");
        j.add_zeros(t[0], extent(t[1]), extent(t[2]), extent(t[3]), extent(t[4]));
    }
    j.run();
    Py_RETURN_NONE;
}

// pools_load(conv pools, ssm pools, K pools, V pools, state conv, state ssm, state kv, slot, pos, Lmax, heads, width)
PyObject* pools_load(PyObject* const* a) {
    const Items pc(a[0]), ps(a[1]), pk(a[2]), pv(a[3]), sc(a[4]), sm(a[5]), kv(a[6]);
    const long slot = integer(a[7]), pos = integer(a[8]), Lmax = integer(a[9]), nkv = integer(a[10]), D = integer(a[11]), par = pos & 1;
    const long C = 3 * CD, N = HV * DV * DK;
    Jobs j;
    j.reserve(2 * sc.size() + 2 * kv.size());
    for (Py_ssize_t i = 0; i < std::min(sc.size(), sm.size()); i++) {
        j.add(pc[i], sc[i], C, (slot * 2 + par) * C, 0, 1, 0, 0);
        j.add(ps[i], sm[i], N, slot * N, 0, 1, 0, 0);
    }
    for (Py_ssize_t i = 0; i < kv.size(); i++) {
        const Items pair(kv[i]);
        if (pair.size() != 2) value_error("state: (K, V) pairs expected");
        const Tensor& K = gpu_tensor(pair[0], "src");
        if (K.dim() != 4) value_error("state: K / V are expected as [1, heads, rows, width]");
        const long smax = K.size(2);
        j.add(pk[i], pair[0], pos * D, slot * nkv * Lmax * D, 0, nkv, Lmax * D, smax * D);
        j.add(pv[i], pair[1], pos * D, slot * nkv * Lmax * D, 0, nkv, Lmax * D, smax * D);
    }
    j.run();
    Py_RETURN_NONE;
}

// element i of the first dimension of a contiguous tensor as a tensor of its own on the same storage
Tensor part_of(const Tensor& t, int64_t i) {
    auto impl = c10::make_intrusive<at::TensorImpl>(c10::Storage(t.storage()), t.key_set(), t.dtype());
    const auto size = t.sizes().slice(1);
    impl->set_sizes_contiguous(size);
    impl->set_storage_offset(t.storage_offset() + i * c10::multiply_integers(size));
    return Tensor(std::move(impl));
}
PyObject* list_of(Py_ssize_t n) {
    PyObject* o = PyList_New(n);
    if (!o) throw Raised{};
    return o;
}
// cache_restore(K / V segments of a checkpoint's chain, conv, ssm, pos, max_len) -> [(K, V)], [conv], [ssm]: the segments [2 layers, 1, heads,
// rows, width] end to end in fresh buffers of max_len rows, rows from pos on zero, and copies of the recurrent state, in one launch
PyObject* cache_restore(PyObject* const* a) {
    const Items segs(a[0]);
    const long pos = integer(a[3]), max_len = integer(a[4]);
    const Tensor &last = gpu_tensor(segs[segs.size() - 1], "kv"), &conv = gpu_tensor(a[1], "conv"), &ssm = gpu_tensor(a[2], "ssm");
    if (last.dim() != 5 || conv.dim() < 1 || ssm.dim() < 1) value_error("cache_restore: kv [2 layers, 1, heads, rows, width] expected");
    const int64_t nb = last.size(0), nkv = last.size(2), D = last.size(4);
    Tensor bufs, conv_out, ssm_out;
    unlocked([&] {
        bufs = empty({nb, 1, nkv, max_len, D}, BF16, last), conv_out = empty(conv.sizes(), conv.scalar_type(), conv), ssm_out = empty(ssm.sizes(), ssm.scalar_type(), ssm);
    });
    Jobs j;
    j.reserve(segs.size() * nb + 3);
    long at = 0;
    for (Py_ssize_t k = 0; k < segs.size(); k++) {
        const Tensor& t = gpu_tensor(segs[k], "kv");
        if (t.dim() != 5 || t.size(0) != nb || t.size(2) != nkv || t.size(4) != D) value_error("cache_restore: the segments' shapes differ");
        const long n = t.size(3);
        for (int64_t i = 0; i < nb; i++) j.add(bufs, segs[k], n * D, i * nkv * max_len * D + at * D, i * nkv * n * D, nkv, max_len * D, n * D);
        at += n;
    }
    if (at != pos) throw Error{PyExc_AssertionError, "cache_restore: " + std::to_string(at) + " rows in the chain, " + std::to_string(pos) + " expected"};
    j.add(conv_out, a[1], conv.numel(), 0, 0, 1, 0, 0);
    j.add(ssm_out, a[2], ssm.numel(), 0, 0, 1, 0, 0);
    if (max_len > pos) j.add_zeros(bufs, (max_len - pos) * D, pos * D, nb * nkv, max_len * D);
    j.run();
    const Ref kv(list_of(nb / 2)), cs(list_of(conv.size(0))), ss(list_of(ssm.size(0)));
    for (int64_t i = 0; i < nb / 2; i++) PyList_SET_ITEM(kv.o, i, wrap({part_of(bufs, 2 * i), part_of(bufs, 2 * i + 1)}));
    for (int64_t i = 0; i < conv.size(0); i++) PyList_SET_ITEM(cs.o, i, wrap(part_of(conv_out, i)));
    for (int64_t i = 0; i < ssm.size(0); i++) PyList_SET_ITEM(ss.o, i, wrap(part_of(ssm_out, i)));
    return PyTuple_Pack(3, kv.o, cs.o, ss.o);
}

// ---- the module -----------------------------------------------------------------------------------------------------------
template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
        return nullptr;
    }
    try {
        return F(args);
    } catch (const Error& e) {
        PyErr_SetString(e.type, e.text.c_str());
    } catch (const Raised&) {
    } catch (const c10::OutOfMemoryError& e) {
        PyObject *torch = PyImport_ImportModule("torch"), *type = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
        if (type) PyErr_SetString(type, e.what_without_backtrace());
        Py_XDECREF(type);
        Py_XDECREF(torch);
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}
#define QT_FN(name, fn, n) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<fn, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    QT_FN("rms_rows", rms_rows, 4),       QT_FN("fused_gemv", fused_gemv, 7),     QT_FN("gated_norm", gated_norm, 4),
    QT_FN("decode_step", decode_step, 9), QT_FN("decode_step_gnorm", decode_step_gnorm, 10), QT_FN("verify_step", verify_step, 11),
    QT_FN("deltanet", deltanet, 8),
    QT_FN("attn_b", attn_b, 10),          QT_FN("attn_layer_b", attn_layer_b, 11), QT_FN("sdpa", sdpa, 3),
    QT_FN("qkv_prep", qkv_prep, 7),       QT_FN("out_gate", out_gate, 2),         QT_FN("conv_prep", conv_prep, 3),
    QT_FN("phase_a", phase_a, 8),         QT_FN("phase_b", phase_b, 5),           QT_FN("phase_b_norm", phase_b_norm, 7),
    QT_FN("gdn_core", gdn_core, 7),
    QT_FN("set_hooks", set_hooks, 3),     QT_FN("blit_batch", blit_batch, 2),     QT_FN("pools_load", pools_load, 12),
    QT_FN("cache_restore", cache_restore, 5),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_qt_host", "argument checks, allocation and launch of the operators", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__qt_host() { return PyModule_Create(&module); }
