// The launchers' steady state in native code (CPython extension _native).
//
// A launch whose tables the Python launchers have checked and planned before costs them 4 to 25 us of host work - argument
// checks, notes about the tables, temporaries, the descriptor - beside the 3 us of the launch itself, which is what small
// steps wait for.  The functions here do that work for ordinary operands and either launch, or return None and touch nothing:
// then the Python launcher goes through its general path, which also raises every error.
//
// What is known about a set of tables is kept here under the conditions of the launchers' own notes: the same tensors, alive
// (weak references), at the same version, and the same sizes and options.  Operands are looked at on every call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <map>
#include <set>
#include <thread>
#include <tuple>
#include <vector>

#include "../../include/syncopate_hip.h"

namespace {

typedef int (*gemm_fn)(const syn_gemm_desc*, syn_stream_t);
typedef int (*remote_fn)(const syn_gemm_desc*, const syn_gemm_remote*, syn_stream_t);
typedef int (*reduce_fn)(const void*, int64_t, const void*, void*, int32_t, int32_t, int64_t, int64_t, int32_t, int32_t,
                         syn_stream_t);
typedef int (*attn_fn)(const syn_attn_desc*, syn_stream_t);
gemm_fn g_consumer = nullptr, g_producer = nullptr;
remote_fn g_remote = nullptr;
reduce_fn g_reduce = nullptr;
attn_fn g_attn = nullptr;
typedef int (*read_fn)(const int32_t* const*, const int32_t*, int32_t, int32_t*, uint64_t*, uint64_t, syn_stream_t);
read_fn g_read = nullptr;

constexpr size_t kMaxRecords = 1024, kMaxPools = 64;
constexpr int kPoolAreas = 16;

// ---------------------------------------------------------------- operands

// A plain tensor in the memory of device `dev` (-1: any), or null.  Subclasses and wrappers, inference tensors (no version)
// and everything under an active dispatch mode take the general path.
const at::Tensor* plain(PyObject* obj, int dev = -1) {
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(obj);
    if (!t.defined() || !t.is_cuda() || t.is_inference() || at::isTensorSubclassLike(t) || t.layout() != at::kStrided ||
        t.is_conj() || t.is_neg())
        return nullptr;
    return dev >= 0 && t.device().index() != dev ? nullptr : &t;
}

bool modes_active() { return c10::impl::TorchDispatchModeTLS::any_modes_set(); }

int dtype_code(const at::Tensor& t) {
    return t.scalar_type() == at::kBFloat16 ? SYN_DTYPE_BF16 : t.scalar_type() == at::kHalf ? SYN_DTYPE_FP16 : -1;
}

bool int_table(const at::Tensor& t, int64_t width) {
    return t.scalar_type() == at::kInt && t.is_contiguous() && (width == 0 ? t.dim() == 1 : t.dim() == 2 && t.size(1) == width);
}

bool flag_words(const at::Tensor& t) {
    return (t.scalar_type() == at::kLong || t.scalar_type() == at::kUInt64) && t.is_contiguous();
}

int64_t as_int(PyObject* obj, bool* ok) {
    const long long v = PyLong_AsLongLong(obj);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        *ok = false;
    }
    return (int64_t)v;
}

int64_t stream_of(int dev) { return reinterpret_cast<int64_t>(c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream()); }

// the launch of `fn` on the current stream, without the interpreter's lock
template <typename F>
int launch(int dev, F&& fn) {
    hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(reinterpret_cast<syn_stream_t>(stream));
    Py_END_ALLOW_THREADS
    return rc;
}

bool capturing(int dev) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
    if (hipStreamIsCapturing(stream, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
    (void)hipGetLastError();             // (the general path asks again, and reports it)
    return true;
}

// ---------------------------------------------------------------- what is known about a set of tables

// A launch is known by its kind, the tables' objects and what `params` lists: sizes, options, for C bound to buffers their addresses,
// and the stream, on which the launcher has marked the device tables that a record keeps as read.
struct Known {
    std::vector<c10::weak_intrusive_ptr<c10::TensorImpl>> tables;
    std::vector<int64_t> versions;
    at::Tensor status;
    std::vector<at::Tensor> keep;            // device tables the descriptor points into
    syn_gemm_desc gemm = {};
    syn_gemm_remote remote = {};
    syn_attn_desc attn = {};
    int64_t lock_words = 0, node_words = 0, partial_bytes = 0;

    // (a weak reference keeps its address from being handed out again: the same address and alive is the same tensor)
    bool alive() const {
        for (const auto& t : tables)
            if (t.expired()) return false;
        return true;
    }
};
typedef std::vector<int64_t> Key;
std::map<Key, Known> g_known;

Key key_of(int64_t kind, const std::vector<const at::Tensor*>& tables, const std::vector<int64_t>& params) {
    Key key;
    key.reserve(1 + tables.size() + params.size());
    key.push_back(kind);
    for (const at::Tensor* t : tables) key.push_back(reinterpret_cast<int64_t>(t->unsafeGetTensorImpl()));
    key.insert(key.end(), params.begin(), params.end());
    return key;
}

const Known* recall(int64_t kind, const std::vector<const at::Tensor*>& tables, const std::vector<int64_t>& params) {
    const auto found = g_known.find(key_of(kind, tables, params));
    if (found == g_known.end() || !found->second.alive()) return nullptr;
    for (size_t i = 0; i < tables.size(); ++i)
        if ((int64_t)tables[i]->_version() != found->second.versions[i]) return nullptr;
    return &found->second;
}

void remember(int64_t kind, const std::vector<const at::Tensor*>& tables, const std::vector<int64_t>& params, Known&& k) {
    for (const at::Tensor* t : tables) {
        k.tables.emplace_back(t->getIntrusivePtr());
        k.versions.push_back((int64_t)t->_version());
    }
    if (g_known.size() >= kMaxRecords) {
        for (auto i = g_known.begin(); i != g_known.end();) i = i->second.alive() ? std::next(i) : g_known.erase(i);
        if (g_known.size() >= kMaxRecords / 4 * 3) g_known.clear();      // (or the next ones would be looked through again soon)
    }
    g_known[key_of(kind, tables, params)] = std::move(k);
}

// ---------------------------------------------------------------- zeroed work areas

// An area of zeros for one launch (see zeroed_int32 of the launchers: one fill kernel for sixteen launches), per thread: between
// taking an area and launching on it no other thread may have the pool filled again.  The tensor is held until the launch
// is queued.
struct Pool {
    at::Tensor areas;
    int used = 0;
};
std::map<std::tuple<int, void*, int64_t, std::thread::id>, Pool> g_pools;

int32_t* zeroed(int dev, int64_t words, at::Tensor* keep) {
    // (the areas outlive the mode that the first launch came in: an inference tensor could not be filled again outside of it)
    const c10::InferenceMode ordinary(false);
    void* stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
    const auto key = std::make_tuple(dev, stream, words, std::this_thread::get_id());
    auto found = g_pools.find(key);
    if (found == g_pools.end()) {
        if (g_pools.size() >= kMaxPools) g_pools.clear();
        found = g_pools.emplace(key, Pool{}).first;
        found->second.areas = at::zeros({kPoolAreas * words}, at::TensorOptions().dtype(at::kInt).device(at::kCUDA, dev));
    } else if (found->second.used >= kPoolAreas) {
        found->second.areas.zero_();
        found->second.used = 0;
    }
    *keep = found->second.areas;
    return keep->data_ptr<int32_t>() + words * found->second.used++;
}

// ---------------------------------------------------------------- module functions

#define NEED(cond)         \
    do {                   \
        if (!(cond)) Py_RETURN_NONE; \
    } while (0)
#define TRY try {
#define CATCH                                     \
    }                                             \
    catch (const std::exception& e) {             \
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what()); \
        return nullptr;                           \
    }

// the operands of a GEMM: a [M, K] and b [N, K] of one 16-bit type, on the current device
struct GemmOperands {
    const at::Tensor *a, *b;
    int dev, dtype;
    int64_t M, N, K;
};
bool gemm_operands(PyObject* pa, PyObject* pb, GemmOperands* g) {
    g->a = plain(pa);
    if (!g->a || modes_active()) return false;
    g->dev = g->a->device().index();
    g->b = plain(pb, g->dev);
    if (!g->b || g->dev != c10::hip::current_device()) return false;
    g->dtype = dtype_code(*g->a);
    if (g->dtype < 0 || g->a->dim() != 2 || g->b->dim() != 2 || g->b->scalar_type() != g->a->scalar_type() ||
        !g->a->is_contiguous() || !g->b->is_contiguous() || g->a->size(1) != g->b->size(1))
        return false;
    g->M = g->a->size(0);
    g->N = g->b->size(0);
    g->K = g->a->size(1);
    return true;
}

// A launch holds for the rule (a function) that chose its kernel tile.  Those that a record was made under are kept, so that another
// one does not come to the same address.
int64_t rule_of(PyObject* rule, bool keep) {
    static auto* const kept = new std::set<PyObject*>;
    if (keep && kept->insert(rule).second) Py_INCREF(rule);
    return reinterpret_cast<int64_t>(rule);
}

// gemm(a, b, c, signal, sizes, offsets, signals, num_sms, bm, bn, bk, group_m, cum_tiles, xcd_remap, rule, producer, acquire
// [, desc, status])
// With a descriptor (bytes) the launch it came from is remembered; else a remembered one is launched.
constexpr int kKindGemm = 0, kKindProducer = 1, kKindRemote = 2, kKindAttn = 3;

PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TRY
    NEED(n == 17 || n == 19);
    GemmOperands g;
    NEED(gemm_operands(args[0], args[1], &g));
    const at::Tensor *c = plain(args[2], g.dev), *flags = plain(args[3], g.dev);
    NEED(c && flags);
    std::vector<const at::Tensor*> tables(3);
    for (int i = 0; i < 3; ++i) {
        tables[i] = plain(args[4 + i], g.dev);
        NEED(tables[i] && int_table(*tables[i], i < 2 ? 2 : 0));
    }
    NEED(c->scalar_type() == g.a->scalar_type() && c->dim() == 2 && c->size(0) == g.M && c->size(1) == g.N && c->is_contiguous());
    NEED(flag_words(*flags));
    bool ok = true;
    const bool producer = as_int(args[15], &ok) != 0, acquire = as_int(args[16], &ok) != 0;
    std::vector<int64_t> params = {g.M, g.N, g.K, g.dtype, g.dev, stream_of(g.dev), flags->numel()};
    params.reserve(18);
    for (int i = 7; i < 14; ++i) params.push_back(as_int(args[i], &ok));
    params.push_back(rule_of(args[14], n == 19));
    NEED(ok);
    for (const at::Tensor* t : tables) params.push_back(t->numel());
    const int kind = producer ? kKindProducer : kKindGemm;
    if (n == 19) {
        const at::Tensor* status = plain(args[18], g.dev);
        NEED(status && PyBytes_Check(args[17]) && PyBytes_GET_SIZE(args[17]) == (Py_ssize_t)sizeof(syn_gemm_desc));
        Known k;
        memcpy(&k.gemm, PyBytes_AS_STRING(args[17]), sizeof k.gemm);
        k.status = *status;
        remember(kind, tables, params, std::move(k));
        Py_RETURN_NONE;
    }
    const Known* k = recall(kind, tables, params);
    NEED(k != nullptr);
    syn_gemm_desc d = k->gemm;
    at::Tensor keep, status = k->status;
    if (producer) {
        NEED(!capturing(g.dev));
        d.counters = zeroed(g.dev, d.num_waves, &keep);
    }
    d.a = g.a->data_ptr();
    d.b = g.b->data_ptr();
    d.c = c->data_ptr();
    d.flags = static_cast<uint64_t*>(flags->data_ptr());
    d.wave_sizes = static_cast<const int32_t*>(tables[0]->data_ptr());
    d.wave_offsets = static_cast<const int32_t*>(tables[1]->data_ptr());
    d.signal_offsets = static_cast<const int32_t*>(tables[2]->data_ptr());
    d.status = static_cast<int32_t*>(status.data_ptr());
    d.options = (d.options & ~SYN_GEMM_ACQUIRE_ALWAYS) | (acquire ? SYN_GEMM_ACQUIRE_ALWAYS : 0);
    const int rc = launch(g.dev, [&](syn_stream_t s) { return producer ? g_producer(&d, s) : g_consumer(&d, s); });
    return PyLong_FromLong(rc);
    CATCH
}

// remote(a, b, c_list, sizes, offsets, target_rank, dst_offsets, num_sms, bm, bn, bk, group_m, cum_tiles, xcd_remap, M, atomic, rule
// [, desc, remote desc, status, kept tensors]): C bound to a list of buffers, no flags to wait for
PyObject* remote(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TRY
    NEED(n == 17 || n == 21);
    GemmOperands g;
    NEED(gemm_operands(args[0], args[1], &g));
    NEED(PyList_CheckExact(args[2]));
    std::vector<const at::Tensor*> tables(4);
    for (int i = 0; i < 4; ++i) {
        tables[i] = plain(args[3 + i], g.dev);
        NEED(tables[i] && int_table(*tables[i], i == 2 ? 0 : 2));
    }
    bool ok = true;
    const Py_ssize_t buffers = PyList_GET_SIZE(args[2]);
    std::vector<int64_t> params = {g.M, g.N, g.K, g.dtype, g.dev, stream_of(g.dev)};
    params.reserve(20 + 3 * (size_t)buffers);
    for (int i = 7; i < 16; ++i) params.push_back(as_int(args[i], &ok));
    NEED(ok && params[13] == g.M);
    params.push_back(rule_of(args[16], n == 21));
    for (const at::Tensor* t : tables) params.push_back(t->numel());
    for (Py_ssize_t i = 0; i < buffers; ++i) {
        const at::Tensor* c = plain(PyList_GET_ITEM(args[2], i), g.dev);
        NEED(c && c->dim() == 2 && c->scalar_type() == g.a->scalar_type() && c->is_contiguous());
        params.push_back(reinterpret_cast<int64_t>(c->data_ptr()));
        params.push_back(c->size(0));
        params.push_back(c->size(1));
    }
    if (n == 21) {
        const at::Tensor* status = plain(args[19], g.dev);
        NEED(status && PyBytes_Check(args[17]) && PyBytes_GET_SIZE(args[17]) == (Py_ssize_t)sizeof(syn_gemm_desc));
        NEED(PyBytes_Check(args[18]) && PyBytes_GET_SIZE(args[18]) == (Py_ssize_t)sizeof(syn_gemm_remote));
        NEED(PyList_CheckExact(args[20]));
        Known k;
        memcpy(&k.gemm, PyBytes_AS_STRING(args[17]), sizeof k.gemm);
        memcpy(&k.remote, PyBytes_AS_STRING(args[18]), sizeof k.remote);
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[20]); ++i) {
            const at::Tensor* t = plain(PyList_GET_ITEM(args[20], i), g.dev);
            NEED(t);
            k.keep.push_back(*t);
        }
        k.status = *status;
        remember(kKindRemote, tables, params, std::move(k));
        Py_RETURN_NONE;
    }
    const Known* k = recall(kKindRemote, tables, params);
    NEED(k != nullptr && !capturing(g.dev));      // (a graph must not point into what a record keeps)
    syn_gemm_desc d = k->gemm;
    syn_gemm_remote r = k->remote;
    const std::vector<at::Tensor> keep = k->keep;
    at::Tensor status = k->status;
    d.a = g.a->data_ptr();
    d.b = g.b->data_ptr();
    d.wave_sizes = static_cast<const int32_t*>(tables[0]->data_ptr());
    d.wave_offsets = static_cast<const int32_t*>(tables[1]->data_ptr());
    r.c_target_rank = static_cast<const int32_t*>(tables[2]->data_ptr());
    r.c_dst_offsets = static_cast<const int32_t*>(tables[3]->data_ptr());
    d.status = static_cast<int32_t*>(status.data_ptr());
    return PyLong_FromLong(launch(g.dev, [&](syn_stream_t s) { return g_remote(&d, &r, s); }));
    CATCH
}

// reduce(input, output, local_output, begin_idx, acc_mode)
PyObject* reduce(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TRY
    NEED(n == 5);
    const at::Tensor* in = plain(args[0]);
    NEED(in && !modes_active());
    const int dev = in->device().index();
    const at::Tensor *out = plain(args[1], dev), *local = plain(args[2], dev);
    NEED(out && local && dev == c10::hip::current_device());
    const int dtype = dtype_code(*in);
    NEED(dtype >= 0 && out->scalar_type() == in->scalar_type() && local->scalar_type() == in->scalar_type());
    NEED(in->dim() == 3 && out->dim() == 2 && local->dim() == 2);
    const int64_t world = in->size(0), rows = in->size(1), cols = in->size(2);
    NEED(out->size(0) == rows && out->size(1) == cols && local->size(0) == world * rows && local->size(1) == cols);
    NEED(world > 1 && out->is_contiguous() && local->is_contiguous() && in->stride(2) == 1 && in->stride(1) == cols &&
         in->stride(0) >= rows * cols);
    bool ok = true;
    const int64_t begin = as_int(args[3], &ok), acc = as_int(args[4], &ok);
    NEED(ok && begin >= INT32_MIN && begin <= INT32_MAX && world <= INT32_MAX);
    const int rc = launch(dev, [&](syn_stream_t s) {
        return g_reduce(in->data_ptr(), in->stride(0), local->data_ptr(), out->data_ptr(), (int32_t)world, (int32_t)begin, rows,
                        cols, dtype, (int32_t)acc, s);
    });
    return PyLong_FromLong(rc);
    CATCH
}

bool attn_strides(const at::Tensor& t, int h_ax, int s_ax, int64_t (&out)[3]) {
    out[0] = t.stride(0);
    out[1] = t.stride(h_ax);
    out[2] = t.stride(s_ax);
    return t.stride(3) == 1 && out[0] % 8 == 0 && out[1] % 8 == 0 && out[2] % 8 == 0;
}

// attention(q, k, v, sm_scale, offsets, sizes, cums, signals, signal_ptr, num_waves, cum_tiles, causal, bshd, auto, counters, out,
// return_lse, acquire[, desc, status, work list, lock words, node words, partial bytes]) -> o, (o, lse), an error code or None
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TRY
    NEED(n == 18 || n == 24);
    const at::Tensor* q = plain(args[0]);
    NEED(q && !modes_active());
    const int dev = q->device().index();
    const at::Tensor *k = plain(args[1], dev), *v = plain(args[2], dev), *flags = plain(args[8], dev);
    NEED(k && v && flags && dev == c10::hip::current_device() && flag_words(*flags));
    const int dtype = dtype_code(*q);
    NEED(dtype >= 0 && k->scalar_type() == q->scalar_type() && v->scalar_type() == q->scalar_type());
    NEED(q->dim() == 4 && k->dim() == 4 && v->dim() == 4 && q->size(3) == 128 && k->size(3) == 128);
    std::vector<const at::Tensor*> tables(4);
    for (int i = 0; i < 4; ++i) {
        tables[i] = plain(args[4 + i], dev);
        NEED(tables[i] && int_table(*tables[i], i < 2 ? 4 : 0));
    }
    bool ok = true;
    std::vector<int64_t> params;
    params.reserve(20);
    for (int i = 9; i < 14; ++i) params.push_back(as_int(args[i], &ok));      // num_waves, cum_tiles, causal, bshd, auto
    const bool return_lse = as_int(args[16], &ok) != 0, acquire = as_int(args[17], &ok) != 0;
    const double scale = PyFloat_AsDouble(args[3]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    NEED(ok);
    const int h_ax = params[3] ? 2 : 1, s_ax = params[3] ? 1 : 2;
    const int64_t Z = q->size(0), H = q->size(h_ax), Sq = q->size(s_ax), Skv = k->size(s_ax);
    NEED(k->size(0) == Z && k->size(h_ax) == H && v->sizes() == k->sizes());
    const at::Tensor* counters = nullptr;
    if (args[14] != Py_None) {
        counters = plain(args[14], dev);
        NEED(counters && counters->scalar_type() == at::kInt && counters->is_contiguous());
    }
    for (const int64_t x : {Z, H, Sq, Skv, flags->numel(), (int64_t)dev, stream_of(dev), (int64_t)(counters != nullptr)}) params.push_back(x);
    for (const at::Tensor* t : tables) params.push_back(t->numel());

    if (n == 24) {
        const at::Tensor* status = plain(args[19], dev);
        NEED(status && PyBytes_Check(args[18]) && PyBytes_GET_SIZE(args[18]) == (Py_ssize_t)sizeof(syn_attn_desc));
        Known r;
        memcpy(&r.attn, PyBytes_AS_STRING(args[18]), sizeof r.attn);
        if (args[20] != Py_None) {
            const at::Tensor* list = plain(args[20], dev);
            NEED(list);
            r.keep.push_back(*list);
        }
        r.lock_words = as_int(args[21], &ok);
        r.node_words = as_int(args[22], &ok);
        r.partial_bytes = as_int(args[23], &ok);
        NEED(ok);
        r.status = *status;
        remember(kKindAttn, tables, params, std::move(r));
        Py_RETURN_NONE;
    }
    const Known* known = recall(kKindAttn, tables, params);
    NEED(known != nullptr);
    syn_attn_desc d = known->attn;
    NEED(counters == nullptr || counters->numel() >= d.num_waves);
    at::Tensor o;
    if (args[15] != Py_None) {
        const at::Tensor* out = plain(args[15], dev);
        NEED(out && out->sizes() == q->sizes() && out->scalar_type() == q->scalar_type());
        o = *out;
        NEED(attn_strides(o, h_ax, s_ax, d.o_strides));
    }
    NEED(attn_strides(*q, h_ax, s_ax, d.q_strides) && attn_strides(*k, h_ax, s_ax, d.k_strides) &&
         attn_strides(*v, h_ax, s_ax, d.v_strides));
    NEED(!capturing(dev));
    const at::Tensor status = known->status;
    const std::vector<at::Tensor> keep = known->keep;
    const int64_t lock_words = known->lock_words, node_words = known->node_words, partial_bytes = known->partial_bytes;
    // (nothing of the record is read from here on: an allocation may run the collector, and with it other launches)
    const auto on_dev = at::TensorOptions().device(at::kCUDA, dev);
    if (!o.defined()) {
        o = at::empty(q->sizes(), on_dev.dtype(q->scalar_type()));
        NEED(attn_strides(o, h_ax, s_ax, d.o_strides));
    }
    const at::Tensor lse = at::empty({Z, H, Sq}, on_dev.dtype(at::kFloat));
    at::Tensor locks, nodes, partials;
    d.lock = d.first = nullptr;
    if (lock_words > 0) {
        d.lock = zeroed(dev, lock_words, &locks);
        d.first = d.lock + lock_words / 2;
    }
    d.split_nodes = node_words > 0 ? zeroed(dev, node_words, &nodes) : nullptr;
    if (partial_bytes > 0) partials = at::empty({partial_bytes}, on_dev.dtype(at::kByte));
    d.split_partials = partial_bytes > 0 ? partials.data_ptr() : nullptr;
    d.work_list = keep.empty() ? nullptr : static_cast<const int32_t*>(keep[0].data_ptr());
    d.q = q->data_ptr();
    d.k = k->data_ptr();
    d.v = v->data_ptr();
    d.o = o.data_ptr();
    d.lse = static_cast<float*>(lse.data_ptr());
    d.flags = static_cast<uint64_t*>(flags->data_ptr());
    d.wave_offsets = static_cast<const int32_t*>(tables[0]->data_ptr());
    d.wave_sizes = static_cast<const int32_t*>(tables[1]->data_ptr());
    d.cum_wave_sizes = static_cast<const int32_t*>(tables[2]->data_ptr());
    d.signal_offsets = static_cast<const int32_t*>(tables[3]->data_ptr());
    d.counters = counters ? static_cast<int32_t*>(counters->data_ptr()) : nullptr;
    d.status = static_cast<int32_t*>(status.data_ptr());
    d.dtype = dtype;
    d.sm_scale = (float)scale;
    d.options = (d.options & ~SYN_ATTN_ACQUIRE_ALWAYS) | (acquire ? SYN_ATTN_ACQUIRE_ALWAYS : 0);
    const int rc = launch(dev, [&](syn_stream_t s) { return g_attn(&d, s); });
    if (rc != 0) return PyLong_FromLong(rc);
    if (!return_lse && args[15] != Py_None) {
        Py_INCREF(args[15]);
        return args[15];
    }
    PyObject* po = args[15] != Py_None ? (Py_INCREF(args[15]), args[15]) : THPVariable_Wrap(o);
    if (!return_lse || !po) return po;
    PyObject* pl = THPVariable_Wrap(lse);
    PyObject* both = pl ? PyTuple_Pack(2, po, pl) : nullptr;
    Py_DECREF(po);
    Py_XDECREF(pl);
    return both;
    CATCH
}

// read_tables(table, ...) -> the words of one to four small int32 tables as bytes, as they are at this point of the current
// stream, or None
//
// The words go to pinned memory that this call has to itself (from a bounded list that is never freed: the process may end
// in any order) and the host looks at the word behind them.  Work in front of it that takes long is waited for asleep.
constexpr int64_t kReadWords = 4096;
PyObject* read_tables(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TRY
    NEED(n >= 1 && n <= 4 && !modes_active());
    const at::Tensor* first = plain(args[0]);
    NEED(first);
    const int dev = first->device().index();
    NEED(dev == c10::hip::current_device() && !capturing(dev));
    const int32_t* tables[4];
    int32_t counts[4];
    int64_t words = 0;
    for (int i = 0; i < (int)n; ++i) {
        const at::Tensor* t = plain(args[i], dev);
        NEED(t && t->scalar_type() == at::kInt && t->is_contiguous() && t->numel() <= kReadWords);
        tables[i] = static_cast<const int32_t*>(t->data_ptr());
        counts[i] = (int32_t)t->numel();
        words += counts[i];
    }
    NEED(words > 0 && words <= kReadWords);
    static auto* const spare = new std::vector<at::Tensor>;
    static uint64_t last = 0;
    at::Tensor buffer;
    if (!spare->empty()) {
        buffer = spare->back();
        spare->pop_back();
    } else {
        buffer = at::zeros({kReadWords + 16}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    }
    int32_t* const out = buffer.data_ptr<int32_t>();
    uint64_t* const flag = reinterpret_cast<uint64_t*>(out + kReadWords);
    const uint64_t seq = ++last;
    hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
    int rc;
    bool there = false;
    Py_BEGIN_ALLOW_THREADS
    rc = g_read(tables, counts, (int32_t)n, out, flag, seq, reinterpret_cast<syn_stream_t>(stream));
    if (rc == 0) {
        for (int i = 0; i < 20000 && !(there = __atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq); ++i) __builtin_ia32_pause();
        if (!there) {
            rc = (int)hipStreamSynchronize(stream);
            there = __atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq;
        }
    }
    Py_END_ALLOW_THREADS
    if (rc != 0 || !there) {                 // (the buffer may still be written to: it is not used again)
        new at::Tensor(buffer);
        PyErr_Format(PyExc_RuntimeError, "reading the wave tables back failed: %d", rc);
        return nullptr;
    }
    PyObject* bytes = PyBytes_FromStringAndSize(reinterpret_cast<const char*>(out), words * 4);
    if (spare->size() < 8) spare->push_back(buffer);
    return bytes;
    CATCH
}

// bind(addresses of syn_gemm_consumer, syn_gemm_producer, syn_gemm_remote_binding, syn_ring_reduce_strided, syn_attn_fwd,
// syn_read_tables_async)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 6) {
        PyErr_SetString(PyExc_TypeError, "bind takes six addresses");
        return nullptr;
    }
    void* fn[6];
    for (int i = 0; i < 6; ++i) {
        fn[i] = PyLong_AsVoidPtr(args[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    g_consumer = reinterpret_cast<gemm_fn>(fn[0]);
    g_producer = reinterpret_cast<gemm_fn>(fn[1]);
    g_remote = reinterpret_cast<remote_fn>(fn[2]);
    g_reduce = reinterpret_cast<reduce_fn>(fn[3]);
    g_attn = reinterpret_cast<attn_fn>(fn[4]);
    g_read = reinterpret_cast<read_fn>(fn[5]);
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, "the library's entry points"},
    {"gemm", (PyCFunction)(void*)gemm, METH_FASTCALL, "launch (or remember) a chunk-scheduled GEMM"},
    {"remote", (PyCFunction)(void*)remote, METH_FASTCALL, "launch (or remember) a GEMM whose C is bound to peers"},
    {"reduce", (PyCFunction)(void*)reduce, METH_FASTCALL, "launch a chunked ring reduce"},
    {"attention", (PyCFunction)(void*)attention, METH_FASTCALL, "launch (or remember) a chunked attention"},
    {"read_tables", (PyCFunction)(void*)read_tables, METH_FASTCALL, "the words of four small tables in device memory"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", "steady-state launches", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&g_module); }
