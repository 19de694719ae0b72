// Host path of the quantized-linear calls: argument checks, allocation and the library call of a
// forward in one native step.
//
// At one token the two launches of a linear take 9 us on the GPU, and the same call through Python
// objects and ctypes took 27-50 us of host time, so eager decoding ran at the host's speed.  Here a
// call costs its two launches and two allocations.  Every function returns None for anything it
// does not recognise -- other tensor types, dispatch or functorch modes, a wrong argument, a size that
// takes the library-GEMM route -- having done nothing; the Python code then serves the call or
// names what is wrong with it.
//
// The library's entry points come from the handle that ctypes opened (`bind`), so both sides always
// call the same build.
#include <Python.h>
#include <dlfcn.h>

#include <algorithm>
#include <array>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/glq_hip.h"

namespace {

struct {
    decltype(&glqh_last_error) last_error;
    decltype(&glqh_fused_linear_trellis_workspace_bytes) trellis_ws;
    decltype(&glqh_fused_linear_trellis_3inst) trellis;
    decltype(&glqh_fused_linear_e8_workspace_bytes) e8_ws;
    decltype(&glqh_fused_linear_e8_folded) e8;
    decltype(&glqh_e8_fold_eligible) fold_eligible;
    decltype(&glqh_e8_few_eligible) few_eligible;
    decltype(&glqh_fused_linear_trellis_group_workspace_bytes) group_ws;
    decltype(&glqh_fused_linear_trellis_3inst_group) group;
    decltype(&glqh_fused_linear_trellis_3inst_group_rvq2) group_rvq2;
    decltype(&glqh_fused_moe_trellis_workspace_bytes) moe_ws;
    decltype(&glqh_fused_moe_trellis_3inst) moe;
    decltype(&glqh_e8_shell_workspace_bytes) shell_ws;
    decltype(&glqh_e8_shell_quantize) shell_quantize;
} L;

PyObject *g_ext = nullptr;                                     // glq_amd.ext's globals: its switches are read per call
PyObject *g_oom = nullptr;                                     // torch.OutOfMemoryError
PyObject *s_buffers, *s_SV, *s_SU, *s_tp, *s_tp2, *s_tlut, *s_bias, *s_codebook, *s_codebook2, *s_shards;
PyObject *s_q[4], *s_dense, *s_fuse, *s_tmax, *s_smax, *s_fold, *s_emax, *s_efmax;

constexpr int64_t MOST_TOKENS = 32768;                         // _MAX_TOKENS_PER_CALL

// ---- tensors --------------------------------------------------------------------------
const c10::DispatchKeySet PLAIN({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA,
                                  c10::DispatchKey::AutocastCUDA});

// An ordinary contiguous GPU tensor of this type, or null.  The pointer is good while this thread has the GIL: a layer's
// buffers can be replaced by another thread once a call gives it up, so what a call reads after that it holds by value.
const at::Tensor *gpu(PyObject *o, at::ScalarType dt) {
    if (!o || !THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || t.scalar_type() != dt || (t.key_set() | PLAIN) != PLAIN || !t.is_cuda() || !t.is_contiguous()) return nullptr;
    if (t.requires_grad() && c10::GradMode::is_enabled()) return nullptr;   // the operators say that they are not differentiable
    return &t;
}

const at::Tensor *activations(PyObject *o) {
    const at::Tensor *t = gpu(o, at::kBFloat16);
    return t ? t : gpu(o, at::kHalf);
}

int lib_type(at::ScalarType t) { return t == at::kHalf ? GLQH_F16 : t == at::kBFloat16 ? GLQH_BF16 : GLQH_F32; }

// a Python dispatch mode, or torch.jit.trace above the dispatcher: the call has to be seen as an operator
bool modes() { return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::tracer::impl::is_dispatch_enabled(); }

bool integer(PyObject *o, int64_t *v) {
    if (!PyLong_CheckExact(o)) return false;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}

bool real(PyObject *o, double *v) {
    if (PyFloat_CheckExact(o)) { *v = PyFloat_AS_DOUBLE(o); return true; }
    int64_t i;
    if (!integer(o, &i)) return false;
    *v = (double)i;
    return true;
}

// block sizes: a CPU int64 tensor or a list of ints
struct blocks {
    int64_t own[64];
    const int64_t *p = nullptr;
    int64_t n = 0;
    bool read(PyObject *o) {
        if (!o) return false;
        if (THPVariable_CheckExact(o)) {
            const at::Tensor &t = THPVariable_Unpack(o);
            if (!t.defined() || !t.is_cpu() || t.scalar_type() != at::kLong || t.dim() != 1 || !t.is_contiguous()) return false;
            p = t.const_data_ptr<int64_t>();
            n = t.numel();
            return n >= 1;
        }
        if (!PyList_CheckExact(o) || PyList_GET_SIZE(o) < 1 || PyList_GET_SIZE(o) > 64) return false;
        n = PyList_GET_SIZE(o);
        for (int64_t i = 0; i < n; ++i)
            if (!integer(PyList_GET_ITEM(o, i), own + i)) return false;
        p = own;
        return true;
    }
};

const glqh_block_meta *meta_ptr(const at::Tensor &t) { return t.defined() ? (const glqh_block_meta *)t.const_data_ptr() : nullptr; }

// undefined tensors are on every device
bool same_device(const at::Tensor &x, std::initializer_list<const at::Tensor *> ts) {
    for (const at::Tensor *t : ts)
        if (t->defined() && t->device() != x.device()) return false;
    return true;
}

int64_t setting(PyObject *name, int64_t otherwise) {
    PyObject *v = PyDict_GetItem(g_ext, name);
    int64_t i;
    if (!v) return otherwise;
    if (v == Py_True || v == Py_False) return v == Py_True;
    return integer(v, &i) ? i : otherwise;
}

// scratch of one call, on the current stream; given back to torch's allocator when the call returns
struct scratch {
    c10::DataPtr p;
    size_t bytes;
    explicit scratch(size_t n) : bytes(std::max<size_t>(n, 256)) { p = c10::GetAllocator(c10::DeviceType::CUDA)->allocate(bytes); }
};

void *stream_of(const at::Tensor &x) { return c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

// x's shape with another last dimension
at::Tensor like(const at::Tensor &x, int64_t last, at::ScalarType dt) {
    c10::SmallVector<int64_t, 5> s(x.sizes().begin(), x.sizes().end());
    s.back() = last;
    return at::Tensor(at::detail::empty_cuda(s, dt, x.device(), std::nullopt));
}

PyObject *failed() {
    PyErr_SetString(PyExc_RuntimeError, L.last_error());
    return nullptr;
}

struct no_gil {
    PyThreadState *s = PyEval_SaveThread();
    ~no_gil() { PyEval_RestoreThread(s); }
};

#define NONE_UNLESS(c) do { if (!(c)) Py_RETURN_NONE; } while (0)

// C++ exceptions (out of memory) as RuntimeError, like torch's own
template <typename F>
PyObject *guarded(F f) {
    try {
        return f();
    } catch (const c10::OutOfMemoryError &e) {
        PyErr_SetString(g_oom ? g_oom : PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const c10::Error &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

// a tensor by value; false where it is not what the call recognises
bool hold(PyObject *o, at::ScalarType dt, at::Tensor *to) {
    const at::Tensor *t = gpu(o, dt);
    if (t) *to = *t;
    return t != nullptr;
}

// the block table of a transform of several blocks
bool hold_meta(PyObject *o, int64_t n_blocks, at::Tensor *to) { return n_blocks <= 1 || hold(o, at::kInt, to); }

// ---- one trellis linear ------------------------------------------------------------------
struct trellis_layer {
    at::Tensor sv, su, packed, packed2;                        // packed2: undefined without a second stage
    at::Tensor bn_meta, bm_meta;                               // undefined for a single block
    const int64_t *bn, *bm;
    int64_t n_bn, n_bm;
    double wscale, inv2;
    int64_t in, out, n_pad, m_pad;
};

PyObject *run_trellis(const at::Tensor &x, const trellis_layer &l, at::ScalarType dt) {
    const int64_t B = x.size(-1) ? x.numel() / x.size(-1) : 0;
    NONE_UNLESS(B >= 1 && B <= MOST_TOKENS);
    NONE_UNLESS(PyDict_GetItem(g_ext, s_dense) == Py_False);
    int64_t most = setting(s_tmax, 0);
    const bool two = l.packed2.defined();
    if (two) most = std::min(most, setting(s_smax, 0));
    NONE_UNLESS(B <= most && l.packed.dim() == 2 && (!two || l.packed2.dim() == 2));
    NONE_UNLESS(same_device(x, {&l.sv, &l.su, &l.packed, &l.packed2, &l.bn_meta, &l.bm_meta}));
    return guarded([&]() -> PyObject * {
        c10::DeviceGuard guard(x.device());
        at::Tensor y = like(x, l.out, dt);
        int rc;
        {
            no_gil unlocked;
            scratch ws(L.trellis_ws(B, l.n_pad, l.m_pad));
            rc = L.trellis(x.const_data_ptr(), lib_type(x.scalar_type()), x.size(-1), B, l.sv.const_data_ptr(), l.su.const_data_ptr(),
                           l.packed.const_data_ptr(), l.packed.size(0), l.packed.size(1),
                           two ? l.packed2.const_data_ptr() : nullptr, two ? l.packed2.size(0) : 0, two ? l.packed2.size(1) : 0, l.bn, l.n_bn, l.bm, l.n_bm, meta_ptr(l.bn_meta),
                           meta_ptr(l.bm_meta), l.wscale, l.inv2,
                           l.in, l.out, l.n_pad, l.m_pad, y.mutable_data_ptr(), lib_type(dt), l.out, nullptr, 0, ws.p.get(), ws.bytes,
                           stream_of(x));
        }
        return rc ? failed() : THPVariable_Wrap(std::move(y));
    });
}

// trellis_linear(x, sv, su, packed, packed2 | None, blocks_n, blocks_m, blocks_n_meta, blocks_m_meta, wscale,
//                inv_resid_scale2, in_features, out_features, n_pad, m_pad, out_dtype | None)
PyObject *py_trellis_linear(PyObject *, PyObject *const *a, Py_ssize_t n) {
    NONE_UNLESS(n == 16 && !modes());
    const at::Tensor *x = activations(a[0]);
    NONE_UNLESS(x && x->dim() == 2);
    trellis_layer l;
    NONE_UNLESS(hold(a[1], at::kHalf, &l.sv) && hold(a[2], at::kHalf, &l.su) && hold(a[3], at::kShort, &l.packed));
    if (a[4] != Py_None) NONE_UNLESS(hold(a[4], at::kShort, &l.packed2) && l.packed2.numel() > 0);
    blocks bn, bm;
    NONE_UNLESS(bn.read(a[5]) && bm.read(a[6]));
    NONE_UNLESS(hold_meta(a[7], bn.n, &l.bn_meta) && hold_meta(a[8], bm.n, &l.bm_meta));
    l.bn = bn.p; l.n_bn = bn.n; l.bm = bm.p; l.n_bm = bm.n;
    NONE_UNLESS(real(a[9], &l.wscale) && real(a[10], &l.inv2) && integer(a[11], &l.in) && integer(a[12], &l.out) &&
                integer(a[13], &l.n_pad) && integer(a[14], &l.m_pad));
    at::ScalarType dt = at::kHalf;
    if (a[15] != Py_None) {
        NONE_UNLESS(THPDtype_Check(a[15]));
        dt = reinterpret_cast<THPDtype *>(a[15])->scalar_type;
        NONE_UNLESS(dt == at::kHalf || dt == at::kBFloat16 || dt == at::kFloat);
    }
    NONE_UNLESS(l.out >= 1);
    return run_trellis(*x, l, dt);
}

// ---- plans: what a layer object's forward needs beside its buffers -------------------------------
enum kind_t { TRELLIS, SHELL, GROUP };

struct shard_t {
    double wscale, inv2;
    int64_t out, m_pad;
};

struct plan_t {
    kind_t kind;
    int64_t in = 0, out = 0, n_pad = 0, m_pad = 0;
    std::vector<int64_t> bn, bm;
    at::Tensor bn_meta, bm_meta;
    double wscale = 0, inv[3] = {0, 0, 0};
    // shell
    int stages = 1;
    PyObject *codebook[2] = {nullptr, nullptr};                // the module's attributes, as they were
    at::Tensor cb[2], table[2], halves[2];
    int64_t cb_version[2] = {0, 0};
    const void *q_data[4] = {};
    int64_t q_version[4] = {};
    bool folded = false;
    std::vector<c10::weak_intrusive_ptr<c10::TensorImpl>> lo, hi;   // weak: releasing them is the cache's decision
    // group
    bool two_stage = false;
    std::vector<shard_t> shards;
};

struct Plan {
    PyObject_HEAD
    vectorcallfunc call;
    plan_t *p;
};

PyObject *item(PyObject *d, PyObject *name) { return PyDict_GetItem(d, name); }

// y + bias in y's place; takes y's reference
PyObject *add_bias(PyObject *y, const at::Tensor &bias) {
    if (!y || y == Py_None || !bias.defined()) return y;
    PyObject *sum = guarded([&]() -> PyObject * {
        c10::NoGradGuard no_grad;
        const at::Tensor &t = THPVariable_Unpack(y);
        t.add_(bias.to(t.scalar_type()));
        return y;
    });
    if (!sum) Py_DECREF(y);                                    // the addition raised
    return sum;
}

// a layer's bias; undefined if it has none
bool hold_bias(PyObject *buffers, at::Tensor *to) {
    PyObject *b = item(buffers, s_bias);
    return !b || b == Py_None || hold(b, at::kHalf, to);
}

PyObject *forward_trellis(const plan_t &p, PyObject *buffers, const at::Tensor &x) {
    PyObject *tlut = item(buffers, s_tlut), *tp2 = item(buffers, s_tp2);
    NONE_UNLESS(tlut && THPVariable_CheckExact(tlut) && THPVariable_Unpack(tlut).numel() == 0);
    trellis_layer l;
    at::Tensor bias;
    NONE_UNLESS(hold(item(buffers, s_SV), at::kHalf, &l.sv) && hold(item(buffers, s_SU), at::kHalf, &l.su) &&
                hold(item(buffers, s_tp), at::kShort, &l.packed) && tp2 && THPVariable_CheckExact(tp2));
    if (THPVariable_Unpack(tp2).numel() > 0) NONE_UNLESS(hold(tp2, at::kShort, &l.packed2));
    NONE_UNLESS(hold_bias(buffers, &bias));
    l.bn = p.bn.data(); l.n_bn = p.bn.size(); l.bm = p.bm.data(); l.n_bm = p.bm.size();
    if (l.n_bn > 1) l.bn_meta = p.bn_meta;
    if (l.n_bm > 1) l.bm_meta = p.bm_meta;
    l.wscale = p.wscale; l.inv2 = l.packed2.defined() ? p.inv[0] : 0.0; l.in = p.in; l.out = p.out; l.n_pad = p.n_pad; l.m_pad = p.m_pad;
    return add_bias(run_trellis(x, l, x.scalar_type()), bias);
}

PyObject *forward_shell(const plan_t &p, PyObject *self, PyObject *buffers, const at::Tensor &x) {
    NONE_UNLESS(item(self, s_codebook) == p.codebook[0] && item(self, s_codebook2) == p.codebook[1]);
    for (int i = 0; i < 2; ++i) NONE_UNLESS(!p.cb[i].defined() || (int64_t)p.cb[i]._version() == p.cb_version[i]);
    at::Tensor q[4], sv, su, bias;
    for (int i = 0; i < 4; ++i)
        NONE_UNLESS(hold(item(buffers, s_q[i]), at::kShort, q + i) && !q[i].is_inference() && q[i].const_data_ptr() == p.q_data[i] &&
                    (int64_t)q[i]._version() == p.q_version[i]);
    NONE_UNLESS(hold(item(buffers, s_SV), at::kHalf, &sv) && hold(item(buffers, s_SU), at::kHalf, &su) && hold_bias(buffers, &bias));
    const int64_t B = x.numel() / p.in;
    NONE_UNLESS(B >= 1 && B <= MOST_TOKENS && q[0].dim() == 2 && q[0].size(0) == p.m_pad && q[0].size(1) * 8 == p.n_pad);
    NONE_UNLESS(same_device(x, {&sv, &su, &q[0], &q[1], &q[2], &q[3], &p.table[0], &p.table[1], &p.bn_meta, &p.bm_meta}));
    // the routes of ext._e8_dense_route: dequantize + library GEMM is Python's
    const int64_t plain_most = setting(s_emax, 0), fold_most = std::max(plain_most, setting(s_efmax, 0));
    glqh_e8_folded f = {};
    std::vector<c10::intrusive_ptr<c10::TensorImpl>> keep;
    bool folded = false;
    bool wants = !(B > fold_most || (B > 16 && p.n_pad % 32 != 0)) && setting(s_fold, 0);
    if (wants && L.fold_eligible(p.m_pad, p.n_pad, B)) NONE_UNLESS(p.folded);
    else wants = wants && p.folded && L.few_eligible(p.m_pad, p.n_pad, B);   // a small layer: on its indices if not prepared
    if (wants) {
        for (int s = 0; s < p.stages; ++s) {
            auto lo = p.lo[s].lock(), hi = p.hi[s].lock();
            NONE_UNLESS(lo && hi);
            f.lo16[s] = (decltype(f.lo16[s] + 0))lo->data();
            f.hi8[s] = (decltype(f.hi8[s] + 0))hi->data();
            keep.push_back(std::move(lo));
            keep.push_back(std::move(hi));
        }
        f.halves1 = p.halves[0].const_data_ptr();
        f.n_halves1 = p.halves[0].size(0);
        if (p.halves[1].defined()) { f.halves2 = p.halves[1].const_data_ptr(); f.n_halves2 = p.halves[1].size(0); }
        folded = true;
    }
    NONE_UNLESS(!(B > (folded ? fold_most : plain_most) || (B > 16 && p.n_pad % (folded ? 32 : 256) != 0)));
    PyObject *y = guarded([&]() -> PyObject * {
        c10::DeviceGuard guard(x.device());
        at::Tensor out = like(x, p.out, x.scalar_type());
        auto stage = [&](int s) { return s < p.stages ? q[s].const_data_ptr() : nullptr; };
        const bool t2 = p.stages >= 2;
        int rc;
        {
            no_gil unlocked;
            scratch ws(L.e8_ws(B, p.n_pad, p.m_pad));
            rc = L.e8(x.const_data_ptr(), lib_type(x.scalar_type()), p.in, B, sv.const_data_ptr(), su.const_data_ptr(), stage(0), stage(1),
                      stage(2), stage(3), (const uint32_t *)p.table[0].const_data_ptr(),
                      t2 ? (const uint32_t *)p.table[1].const_data_ptr() : nullptr, t2 ? p.table[1].size(0) : 0, p.wscale, p.inv[0],
                      p.inv[1], p.inv[2], p.bn.data(), p.bn.size(), p.bm.data(), p.bm.size(),
                      p.bn.size() > 1 ? meta_ptr(p.bn_meta) : nullptr, p.bm.size() > 1 ? meta_ptr(p.bm_meta) : nullptr, p.in, p.out,
                      p.n_pad, p.m_pad, out.mutable_data_ptr(), lib_type(x.scalar_type()), p.out, ws.p.get(), ws.bytes, stream_of(x),
                      folded ? &f : nullptr);
        }
        return rc ? failed() : THPVariable_Wrap(std::move(out));
    });
    return add_bias(y, bias);
}

// the list behind a GLQShards attribute of a merged layer
PyObject *shard_list(PyObject *self, PyObject *name, size_t n) {
    PyObject *o = item(self, name);
    PyObject **d = o ? _PyObject_GetDictPtr(o) : nullptr;
    PyObject *l = d && *d ? item(*d, s_shards) : nullptr;
    return l && PyList_CheckExact(l) && (size_t)PyList_GET_SIZE(l) == n ? l : nullptr;
}

PyObject *forward_group(const plan_t &p, PyObject *self, const at::Tensor &x) {
    const size_t n = p.shards.size();
    const int64_t B = x.numel() / p.in;
    NONE_UNLESS(B >= 1 && B <= MOST_TOKENS);
    // stacked shards at many tokens: the conditions of MergedTrellisLinear._grouped_rvq2_many_ok
    if (p.two_stage && B > 64)
        NONE_UNLESS(B <= std::min(setting(s_tmax, 0), setting(s_smax, 0)) && PyDict_GetItem(g_ext, s_dense) == Py_False &&
                    PyDict_GetItem(g_ext, s_fuse) == Py_True);
    PyObject *svs = shard_list(self, s_SV, n), *sus = shard_list(self, s_SU, n), *ps = shard_list(self, s_tp, n), *ps2 = shard_list(self, s_tp2, n);
    NONE_UNLESS(svs && sus && ps && ps2 && (p.bn.size() <= 1 || same_device(x, {&p.bn_meta})));
    glqh_trellis_shard sh[GLQH_MAX_SHARDS] = {};
    glqh_trellis_stage2 s2[GLQH_MAX_SHARDS] = {};
    int64_t total_out = 0, total_m = 0;
    std::array<at::Tensor, 4 * GLQH_MAX_SHARDS> keep;          // the lists can change once the GIL is given up
    size_t kept = 0;
    for (size_t i = 0; i < n; ++i) {
        const at::Tensor *sv = gpu(PyList_GET_ITEM(svs, i), at::kHalf), *su = gpu(PyList_GET_ITEM(sus, i), at::kHalf);
        const at::Tensor *pk = gpu(PyList_GET_ITEM(ps, i), at::kShort);
        NONE_UNLESS(sv && su && pk && pk->dim() == 2 && pk->numel() > 0 && same_device(x, {sv, su, pk}));
        for (const at::Tensor *t : {sv, su, pk}) keep[kept++] = *t;
        sh[i] = {sv->const_data_ptr(), su->const_data_ptr(), pk->const_data_ptr(), pk->size(0), pk->size(1), p.shards[i].wscale,
                 p.shards[i].out, p.shards[i].m_pad, nullptr};
        NONE_UNLESS(sh[i].packed_cols == sh[0].packed_cols);
        if (p.two_stage) {
            const at::Tensor *pk2 = gpu(PyList_GET_ITEM(ps2, i), at::kShort);
            NONE_UNLESS(pk2 && pk2->dim() == 2 && pk2->numel() > 0 && same_device(x, {pk2}));
            keep[kept++] = *pk2;
            s2[i] = {pk2->const_data_ptr(), pk2->size(0), pk2->size(1), p.shards[i].inv2};
            NONE_UNLESS(sh[i].packed_cols == 64 && s2[i].packed2_cols == s2[0].packed2_cols);
        }
        total_out += p.shards[i].out;
        total_m += p.shards[i].m_pad;
    }
    return guarded([&]() -> PyObject * {
        c10::DeviceGuard guard(x.device());
        at::Tensor y = like(x, total_out, x.scalar_type());
        int64_t off = 0;
        for (size_t i = 0; i < n; ++i) {
            sh[i].y = (char *)y.mutable_data_ptr() + 2 * off;
            off += p.shards[i].out;
        }
        const glqh_block_meta *bm = p.bn.size() > 1 ? meta_ptr(p.bn_meta) : nullptr;
        int rc;
        {
            no_gil unlocked;
            scratch ws(L.group_ws(B, p.n_pad, total_m, (int)n));
            const int dt = lib_type(x.scalar_type());
            rc = p.two_stage ? L.group_rvq2(x.const_data_ptr(), dt, p.in, B, sh, s2, (int)n, p.bn.data(), p.bn.size(), bm, p.in, p.n_pad, dt,
                                            total_out, ws.p.get(), ws.bytes, stream_of(x))
                             : L.group(x.const_data_ptr(), dt, p.in, B, sh, (int)n, p.bn.data(), p.bn.size(), bm, p.in, p.n_pad, dt,
                                       total_out, ws.p.get(), ws.bytes, stream_of(x));
        }
        return rc ? failed() : THPVariable_Wrap(std::move(y));
    });
}

// plan(layer.__dict__, x)
PyObject *plan_call(PyObject *self, PyObject *const *a, size_t nargs, PyObject *kw) {
    NONE_UNLESS(PyVectorcall_NARGS(nargs) == 2 && !kw && PyDict_CheckExact(a[0]) && !modes());
    const plan_t &p = *((Plan *)self)->p;
    const at::Tensor *given = activations(a[1]);
    NONE_UNLESS(given && given->dim() >= 1 && given->size(-1) == p.in && given->numel() > 0);
    const at::Tensor x = *given;
    if (p.kind == GROUP) return forward_group(p, a[0], x);
    PyObject *buffers = item(a[0], s_buffers);
    NONE_UNLESS(buffers && PyDict_Check(buffers));
    return p.kind == TRELLIS ? forward_trellis(p, buffers, x) : forward_shell(p, a[0], buffers, x);
}

void plan_free(PyObject *self) {
    plan_t *p = ((Plan *)self)->p;
    if (p) {
        Py_XDECREF(p->codebook[0]);
        Py_XDECREF(p->codebook[1]);
        delete p;
    }
    Py_TYPE(self)->tp_free(self);
}

// copies and pickles of a layer make their own plan
PyObject *plan_reduce(PyObject *, PyObject *) { return Py_BuildValue("(O())", (PyObject *)Py_TYPE(Py_None)); }

PyMethodDef plan_methods[] = {{"__reduce__", plan_reduce, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0)};

Plan *new_plan(kind_t kind) {
    Plan *o = PyObject_New(Plan, &PlanType);
    if (!o) return nullptr;
    o->call = plan_call;
    o->p = new plan_t;
    o->p->kind = kind;
    return o;
}

bool list_of(PyObject *o, std::vector<int64_t> *v) {
    blocks b;
    if (!b.read(o)) return false;
    v->assign(b.p, b.p + b.n);
    return true;
}

at::Tensor tensor(PyObject *o) { return o && THPVariable_Check(o) ? THPVariable_Unpack(o) : at::Tensor(); }

PyObject *bad(Plan *o, const char *what) {
    Py_DECREF(o);
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, what);
    return nullptr;
}

// trellis_plan(in, out, n_pad, m_pad, blocks_n, blocks_m, blocks_n_meta, blocks_m_meta, wscale, inv_resid_scale2)
PyObject *py_trellis_plan(PyObject *, PyObject *args) {
    Plan *o = new_plan(TRELLIS);
    if (!o) return nullptr;
    plan_t &p = *o->p;
    PyObject *bn, *bm, *bnm, *bmm;
    if (!PyArg_ParseTuple(args, "LLLLOOOOdd", &p.in, &p.out, &p.n_pad, &p.m_pad, &bn, &bm, &bnm, &bmm, &p.wscale, &p.inv[0]) ||
        !list_of(bn, &p.bn) || !list_of(bm, &p.bm))
        return bad(o, "trellis_plan: block sizes");
    p.bn_meta = tensor(bnm);
    p.bm_meta = tensor(bmm);
    return (PyObject *)o;
}

// shell_plan(in, out, n_pad, m_pad, blocks_n, blocks_m, blocks_n_meta, blocks_m_meta, wscale, inv1, inv2, inv3, stages,
//            codebook, codebook2, cb, cb2 | None, table, table2 | None, [Qidxs x 4], [(lo16, hi8) ...] | None, halves, halves2)
PyObject *py_shell_plan(PyObject *, PyObject *args) {
    Plan *o = new_plan(SHELL);
    if (!o) return nullptr;
    plan_t &p = *o->p;
    PyObject *bn, *bm, *bnm, *bmm, *c1, *c2, *cb1, *cb2, *t1, *t2, *q, *st, *h1, *h2;
    if (!PyArg_ParseTuple(args, "LLLLOOOOddddiOOOOOOOOOO", &p.in, &p.out, &p.n_pad, &p.m_pad, &bn, &bm, &bnm, &bmm, &p.wscale, &p.inv[0],
                          &p.inv[1], &p.inv[2], &p.stages, &c1, &c2, &cb1, &cb2, &t1, &t2, &q, &st, &h1, &h2) ||
        !list_of(bn, &p.bn) || !list_of(bm, &p.bm))
        return bad(o, "shell_plan: block sizes");
    p.bn_meta = tensor(bnm);
    p.bm_meta = tensor(bmm);
    p.codebook[0] = Py_NewRef(c1);
    p.codebook[1] = Py_NewRef(c2);
    p.cb[0] = tensor(cb1); p.cb[1] = tensor(cb2); p.table[0] = tensor(t1); p.table[1] = tensor(t2);
    p.halves[0] = tensor(h1); p.halves[1] = tensor(h2);
    if (p.stages < 1 || p.stages > 4 || !p.table[0].defined() || (p.stages > 1 && !p.table[1].defined()) || !PyList_CheckExact(q) ||
        PyList_GET_SIZE(q) != 4)
        return bad(o, "shell_plan: stages and tables");
    for (int i = 0; i < 2; ++i)
        if (p.cb[i].defined()) {
            if (p.cb[i].is_inference()) return bad(o, "shell_plan: table without a version");
            p.cb_version[i] = p.cb[i]._version();
        }
    for (int i = 0; i < 4; ++i) {
        const at::Tensor t = tensor(PyList_GET_ITEM(q, i));
        if (!t.defined() || t.is_inference()) return bad(o, "shell_plan: indices");
        p.q_data[i] = t.const_data_ptr();
        p.q_version[i] = t._version();
    }
    if (PyList_CheckExact(st) && PyList_GET_SIZE(st) == p.stages && p.halves[0].defined()) {
        for (int i = 0; i < p.stages; ++i) {
            PyObject *pair = PyList_GET_ITEM(st, i);
            const at::Tensor lo = PyTuple_Check(pair) ? tensor(PyTuple_GET_ITEM(pair, 0)) : at::Tensor();
            const at::Tensor hi = PyTuple_Check(pair) ? tensor(PyTuple_GET_ITEM(pair, 1)) : at::Tensor();
            if (!lo.defined() || !hi.defined()) return bad(o, "shell_plan: folded streams");
            p.lo.emplace_back(lo.getIntrusivePtr());
            p.hi.emplace_back(hi.getIntrusivePtr());
        }
        p.folded = true;
    }
    return (PyObject *)o;
}

// group_plan(in, n_pad, blocks_n, blocks_n_meta, [(wscale, inv_resid_scale2, out, m_pad) ...], two_stage)
PyObject *py_group_plan(PyObject *, PyObject *args) {
    Plan *o = new_plan(GROUP);
    if (!o) return nullptr;
    plan_t &p = *o->p;
    PyObject *bn, *bnm, *shards;
    int two;
    if (!PyArg_ParseTuple(args, "LLOOOp", &p.in, &p.n_pad, &bn, &bnm, &shards, &two) || !list_of(bn, &p.bn) || !PyList_CheckExact(shards) ||
        PyList_GET_SIZE(shards) < 1 || PyList_GET_SIZE(shards) > GLQH_MAX_SHARDS)
        return bad(o, "group_plan: shards");
    p.bn_meta = tensor(bnm);
    p.two_stage = two;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(shards); ++i) {
        shard_t s;
        if (!PyArg_ParseTuple(PyList_GET_ITEM(shards, i), "ddLL", &s.wscale, &s.inv2, &s.out, &s.m_pad)) return bad(o, "group_plan: shard");
        p.shards.push_back(s);
    }
    return (PyObject *)o;
}

// ---- routed experts ------------------------------------------------------------------------
// one projection from its six tensors and its sizes
bool projection(PyObject *const *t, const at::Tensor &x, const blocks &bn, const blocks &bm, PyObject *bnm, int64_t in, int64_t out,
                int64_t n_pad, int64_t m_pad, glqh_moe_proj *w) {
    const at::Tensor *pk = gpu(t[0], at::kShort), *su = gpu(t[2], at::kHalf), *sv = gpu(t[3], at::kHalf), *ws = gpu(t[4], at::kFloat);
    if (!pk || !su || !sv || !ws || pk->dim() != 3 || !same_device(x, {pk, su, sv, ws})) return false;
    const int64_t E = pk->size(0);
    if (su->dim() != 2 || su->size(0) != E || su->size(1) != m_pad || sv->numel() != n_pad || ws->numel() != E) return false;
    *w = {};
    if (t[1] != Py_None) {
        if (!THPVariable_CheckExact(t[1])) return false;
        if (THPVariable_Unpack(t[1]).numel() > E) {            // more than the (E, 1, 1) placeholder
            const at::Tensor *p2 = gpu(t[1], at::kShort), *irs = gpu(t[5], at::kFloat);
            if (!p2 || !irs || p2->dim() != 3 || p2->size(0) != E || p2->size(1) != pk->size(1) || irs->numel() != E ||
                !same_device(x, {p2, irs}))
                return false;
            w->packed2 = p2->const_data_ptr();
            w->packed2_cols = p2->size(2);
            w->inv_rs2_dev = irs->const_data_ptr<float>();
        }
    }
    at::Tensor bmeta;                                          // the caller's argument keeps it
    if (!hold_meta(bnm, bn.n, &bmeta) || !same_device(x, {&bmeta})) return false;
    w->packed = pk->const_data_ptr(); w->packed_rows = pk->size(1); w->packed_cols = pk->size(2);
    w->su_f16 = su->const_data_ptr(); w->sv_f16 = sv->const_data_ptr(); w->wscale_dev = ws->const_data_ptr<float>();
    w->blocks_n = bn.p; w->n_blocks_n = bn.n; w->bn_meta_dev = meta_ptr(bmeta); w->blocks_m = bm.p; w->n_blocks_m = bm.n;
    w->in_features = in; w->out_features = out; w->n_pad = n_pad; w->m_pad = m_pad;
    return true;
}

// moe(x, topk_ids, topk_weights, w13 x 6, w2 x 6, hidden, intermediate, w13_out, n_pad13, m_pad13, n_pad2, m_pad2,
//     blocks_n13, blocks_m13, blocks_n13_meta, blocks_m13_meta, the same for w2, activation, out_dtype | None)
PyObject *py_moe(PyObject *, PyObject *const *a, Py_ssize_t n) {
    NONE_UNLESS(n == 32 && !modes());
    const at::Tensor *x = activations(a[0]), *ids = gpu(a[1], at::kLong), *tw = gpu(a[2], at::kFloat);
    NONE_UNLESS(x && ids && tw && x->dim() == 2 && ids->dim() == 2 && ids->sizes() == tw->sizes() && ids->size(0) == x->size(0));
    int64_t v[7], act;
    for (int i = 0; i < 7; ++i) NONE_UNLESS(integer(a[15 + i], v + i));
    NONE_UNLESS(integer(a[30], &act) && act >= 0 && act <= 2 && x->size(1) == v[0] && x->numel() > 0 && ids->numel() > 0);
    blocks bn13, bm13, bn2, bm2;
    NONE_UNLESS(bn13.read(a[22]) && bm13.read(a[23]) && bn2.read(a[26]) && bm2.read(a[27]));
    glqh_moe_proj w13, w2;
    NONE_UNLESS(projection(a + 3, *x, bn13, bm13, a[24], v[0], v[2], v[3], v[4], &w13));
    NONE_UNLESS(projection(a + 9, *x, bn2, bm2, a[28], v[1], v[0], v[5], v[6], &w2));
    NONE_UNLESS(same_device(*x, {ids, tw}));
    at::ScalarType dt = x->scalar_type();
    if (a[31] != Py_None) {
        NONE_UNLESS(THPDtype_Check(a[31]));
        dt = reinterpret_cast<THPDtype *>(a[31])->scalar_type;
        NONE_UNLESS(dt == at::kHalf || dt == at::kBFloat16);
    }
    const int64_t T = ids->size(0), K = ids->size(1), E = THPVariable_Unpack(a[3]).size(0);
    return guarded([&]() -> PyObject * {
        c10::DeviceGuard guard(x->device());
        at::Tensor out = like(*x, v[0], dt);
        int rc;
        {
            no_gil unlocked;
            scratch ws(L.moe_ws(T, K, E, &w13, &w2));
            rc = L.moe(x->const_data_ptr(), lib_type(x->scalar_type()), v[0], T, ids->const_data_ptr<int64_t>(),
                       tw->const_data_ptr<float>(), K, E, &w13, &w2, v[1], (int)act, out.mutable_data_ptr(), lib_type(dt), v[0],
                       ws.p.get(), ws.bytes, stream_of(*x));
        }
        return rc ? failed() : THPVariable_Wrap(std::move(out));
    });
}

// ---- E8 codewords ----------------------------------------------------------------------------
// shell_quantize(x, table, norms, return_decoded) -> (decoded | None, indices)
PyObject *py_shell_quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    NONE_UNLESS(n == 4 && !modes());
    const at::Tensor *x = gpu(a[0], at::kFloat), *table = gpu(a[1], at::kFloat), *norms = gpu(a[2], at::kFloat);
    NONE_UNLESS(x && table && norms && x->dim() == 2 && x->size(1) == 8 && x->size(0) >= 1 && table->dim() == 2 && table->size(1) == 8);
    NONE_UNLESS(table->size(0) <= 65536 && norms->numel() == table->size(0) && same_device(*x, {table, norms}));
    const int decoded = PyObject_IsTrue(a[3]);
    NONE_UNLESS(decoded >= 0);
    const int64_t N = x->size(0);
    return guarded([&]() -> PyObject * {
        c10::DeviceGuard guard(x->device());
        at::Tensor idx(at::detail::empty_cuda({N}, at::kLong, x->device(), std::nullopt)), dec;
        if (decoded) dec = like(*x, 8, at::kFloat);
        int rc;
        {
            no_gil unlocked;
            scratch ws(L.shell_ws(N));
            rc = L.shell_quantize(x->const_data_ptr<float>(), N, table->const_data_ptr<float>(), norms->const_data_ptr<float>(), table->size(0),
                                  idx.mutable_data_ptr<int64_t>(), decoded ? dec.mutable_data_ptr<float>() : nullptr, ws.p.get(),
                                  ws.bytes, stream_of(*x));
        }
        if (rc) return failed();
        return Py_BuildValue("(NN)", decoded ? THPVariable_Wrap(std::move(dec)) : Py_NewRef(Py_None), THPVariable_Wrap(std::move(idx)));
    });
}

// ---- module ------------------------------------------------------------------------------------
// bind(handle of the library, glq_amd.ext's globals)
PyObject *py_bind(PyObject *, PyObject *args) {
    unsigned long long handle;
    PyObject *ext;
    if (!PyArg_ParseTuple(args, "KO!", &handle, &PyDict_Type, &ext)) return nullptr;
    auto sym = [&](auto &f, const char *name) {
        f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(dlsym((void *)(uintptr_t)handle, name));
        if (!f && !PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "the library has no %s", name);
    };
    sym(L.last_error, "glqh_last_error");
    sym(L.trellis_ws, "glqh_fused_linear_trellis_workspace_bytes");
    sym(L.trellis, "glqh_fused_linear_trellis_3inst");
    sym(L.e8_ws, "glqh_fused_linear_e8_workspace_bytes");
    sym(L.e8, "glqh_fused_linear_e8_folded");
    sym(L.fold_eligible, "glqh_e8_fold_eligible");
    sym(L.few_eligible, "glqh_e8_few_eligible");
    sym(L.group_ws, "glqh_fused_linear_trellis_group_workspace_bytes");
    sym(L.group, "glqh_fused_linear_trellis_3inst_group");
    sym(L.group_rvq2, "glqh_fused_linear_trellis_3inst_group_rvq2");
    sym(L.moe_ws, "glqh_fused_moe_trellis_workspace_bytes");
    sym(L.moe, "glqh_fused_moe_trellis_3inst");
    sym(L.shell_ws, "glqh_e8_shell_workspace_bytes");
    sym(L.shell_quantize, "glqh_e8_shell_quantize");
    if (PyErr_Occurred()) return nullptr;
    if (!g_oom) {
        PyObject *torch = PyImport_ImportModule("torch");
        if (!torch) return nullptr;
        g_oom = PyObject_GetAttrString(torch, "OutOfMemoryError");
        Py_DECREF(torch);
        if (!g_oom) PyErr_Clear();
    }
    Py_XSETREF(g_ext, Py_NewRef(ext));
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, "bind(library handle, globals of glq_amd.ext)"},
    {"trellis_linear", (PyCFunction)(void *)py_trellis_linear, METH_FASTCALL, "fused trellis linear, or None"},
    {"moe", (PyCFunction)(void *)py_moe, METH_FASTCALL, "routed trellis experts, or None"},
    {"shell_quantize", (PyCFunction)(void *)py_shell_quantize, METH_FASTCALL, "codewords of a table that may be the shell table, or None"},
    {"trellis_plan", py_trellis_plan, METH_VARARGS, "forward of a trellis E8RHTLinear"},
    {"shell_plan", py_shell_plan, METH_VARARGS, "forward of a shell E8RHTLinear"},
    {"group_plan", py_group_plan, METH_VARARGS, "forward of a merged trellis layer"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_glq_host", "Native host path of glq_amd.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__glq_host(void) {
    PlanType.tp_name = "glq_amd._glq_host.Plan";
    PlanType.tp_basicsize = sizeof(Plan);
    PlanType.tp_dealloc = plan_free;
    PlanType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    PlanType.tp_vectorcall_offset = offsetof(Plan, call);
    PlanType.tp_call = PyVectorcall_Call;
    PlanType.tp_methods = plan_methods;
    if (PyType_Ready(&PlanType) < 0) return nullptr;
    struct { PyObject **p; const char *s; } names[] = {
        {&s_buffers, "_buffers"}, {&s_SV, "SV"}, {&s_SU, "SU"}, {&s_tp, "trellis_packed"}, {&s_tp2, "trellis_packed2"},
        {&s_tlut, "tlut"}, {&s_bias, "bias"}, {&s_codebook, "codebook"}, {&s_codebook2, "codebook2"}, {&s_shards, "_shard_data"},
        {&s_q[0], "Qidxs"}, {&s_q[1], "Qidxs2"}, {&s_q[2], "Qidxs3"}, {&s_q[3], "Qidxs4"}, {&s_dense, "TRELLIS_DENSE"},
        {&s_fuse, "TRELLIS_FUSE_STAGES"}, {&s_tmax, "TRELLIS_BATCH_MAX"}, {&s_smax, "TRELLIS_STACKED_BATCH_MAX"}, {&s_fold, "E8_FOLD"}, {&s_emax, "E8_BATCH_MAX"},
        {&s_efmax, "E8_FOLD_BATCH_MAX"}};
    for (auto &n : names)
        if (!(*n.p = PyUnicode_InternFromString(n.s))) return nullptr;
    return PyModule_Create(&module);
}
