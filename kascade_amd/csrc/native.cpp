// Host side of the per-layer calls: what a layer of a decode step or of a prompt does between Python
// and the kernels -- shape checks, split counts, scratch and outputs from torch's allocator, the C
// ABI call on the current stream -- in one call.  The same steps as Python cost 20 to 35 us per layer,
// several times what the layer's kernels take on short contexts.
//
// Positional arguments only (vectorcall); tensors are torch tensors.  Errors raise KascadeError.  The
// arguments are read with the interpreter lock held; it is released while memory is taken from the
// allocator (which may wait for the device) and the kernels are launched.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include <map>
#include <string>

#include "../../include/kascade_hip.h"

namespace {

PyObject *g_error = nullptr, *g_raw_stream = nullptr, *g_capturing = nullptr;

struct Fail {};                             // a Python error is set
struct Refused { std::string message; };    // becomes a KascadeError; thrown with or without the lock

[[noreturn]] void fail(const char* fmt, ...) {
    char text[1100];   // the library's own messages have up to 1023 characters
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(text, sizeof(text), fmt, ap);
    va_end(ap);
    throw Refused{text};
}

// Without the interpreter lock until the end of the scope.
class Unlocked {
    PyThreadState* state = PyEval_SaveThread();
public:
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    Unlocked& operator=(const Unlocked&) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};

void need(bool ok, const char* msg) {
    if (!ok) fail("%s", msg);
}

void check(int rc) {
    if (rc != 0) fail("%s", kascade_get_last_error());
}

const at::Tensor& tensor(PyObject* o, const char* name) {
    if (!THPVariable_Check(o)) fail("%s must be a tensor", name);
    return THPVariable_Unpack(o);
}

// Device tensor of a given type, contiguous.
const at::Tensor& dense(PyObject* o, at::ScalarType type, const char* name) {
    const at::Tensor& t = tensor(o, name);
    if (!t.is_cuda()) fail("%s must be a device tensor", name);
    if (t.scalar_type() != type) fail("%s must be %s, got %s", name, at::toString(type), at::toString(t.scalar_type()));
    if (!t.is_contiguous()) fail("%s must be contiguous", name);
    return t;
}

long long integer(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw Fail{};
    return v;
}

double number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw Fail{};
    return v;
}

bool truth(PyObject* o) { return PyObject_IsTrue(o) == 1; }

int device_of_caller() {
    static const c10::impl::VirtualGuardImpl impl(c10::DeviceType::CUDA);
    return impl.getDevice().index();
}

// Handle of the current stream of the current device.
void* stream_of(int device) {
    PyObject* d = PyLong_FromLong(device);
    PyObject* s = PyObject_CallOneArg(g_raw_stream, d);
    Py_DECREF(d);
    if (!s) throw Fail{};
    void* p = PyLong_AsVoidPtr(s);
    Py_DECREF(s);
    return p;
}

kascade_half* half_ptr(const at::Tensor& t) { return static_cast<kascade_half*>(t.data_ptr()); }
int32_t* int_ptr(const at::Tensor& t) { return static_cast<int32_t*>(t.data_ptr()); }
float* float_ptr(const at::Tensor& t) { return static_cast<float*>(t.data_ptr()); }

// A model's shape, from query heads, KV heads, head dimension and the tensors' types.
kascade_shape model_shape(const at::Tensor& q, const at::Tensor& k, int64_t heads, int64_t groups, int64_t dim) {
    const at::ScalarType t = q.scalar_type();
    if ((t != at::kHalf && t != at::kBFloat16) || k.scalar_type() != t)
        fail("Q and K must both be float16 or bfloat16, got %s / %s", at::toString(t), at::toString(k.scalar_type()));
    if (dim != 64 && dim != 128) fail("head_dim must be 64 or 128, got %lld", (long long)dim);
    if (groups < 1 || heads % groups || heads / groups < 1 || heads / groups > 16)
        fail("need 1 to 16 query heads per KV head, got %lld query / %lld KV heads", (long long)heads, (long long)groups);
    return kascade_shape{(int32_t)groups, (int32_t)dim, t == at::kBFloat16 ? KASCADE_BF16 : KASCADE_F16,
                         (int32_t)(heads / groups)};
}

at::Tensor empty_like_type(at::IntArrayRef size, const at::Tensor& like, at::ScalarType type) {
    return at::empty(size, like.options().dtype(type));
}

// What kernels.default_num_split takes by default: two workgroups per compute unit, 512 rows each.
int num_split(int64_t lists, double rows, double cap_rows) {
    const int cus = kascade_device_cu_count();
    return kascade_decode_num_split_equal((int)lists, rows, cus > 0 ? cus : 256, 2, 512, cap_rows);
}

// Arrival counters of the fused split merge: zero when made, and zero again after every launch, so
// that launches on one stream share them; one array per stream.
struct Counters {
    PyObject_HEAD
    std::map<void*, at::Tensor>* by_stream;
};

PyObject* counters_new(PyTypeObject* type, PyObject*, PyObject*) {
    Counters* c = reinterpret_cast<Counters*>(type->tp_alloc(type, 0));
    if (c) c->by_stream = new std::map<void*, at::Tensor>;
    return reinterpret_cast<PyObject*>(c);
}
void counters_dealloc(PyObject* o) {
    delete reinterpret_cast<Counters*>(o)->by_stream;
    Py_TYPE(o)->tp_free(o);
}
PyTypeObject CountersType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// With the lock held, which also orders threads that share the object; two that miss at once make an array
// each, and the later one stays.
at::Tensor counters_for(PyObject* o, void* stream, int64_t n, const at::Tensor& like) {
    if (Py_TYPE(o) != &CountersType) fail("expected a _native.Counters object");
    PyObject* c = PyObject_CallNoArgs(g_capturing);
    if (!c) throw Fail{};
    const bool capturing = PyObject_IsTrue(c) == 1;
    Py_DECREF(c);
    const auto options = like.options().dtype(at::kInt);
    // A graph replays on any stream and outlives this object: counters of its own, from its memory pool.
    auto zeros = [&](int64_t size) {
        Unlocked unlocked;
        return at::zeros({size}, options);
    };
    if (capturing) return zeros(n);
    auto& map = *reinterpret_cast<Counters*>(o)->by_stream;
    auto it = map.find(stream);
    if (it != map.end() && it->second.numel() >= n && it->second.device() == like.device()) return it->second;
    const at::Tensor t = zeros(std::max<int64_t>(n, 1024));
    if (map.size() >= 16) map.clear();   // a program that keeps making streams
    map[stream] = t;
    return t;
}

// ------------------------------------------------------------------ transformers tensors
// q [B,H,n,D], k/v [B,G,L,D] with a contiguous last dimension, as strides of [B,tokens,heads,D].
struct HfTensors {
    at::Tensor q, k, v;
    int64_t B, H, n, D, G, L;
    kascade_shape shape;
    static kascade_strides strides(const at::Tensor& t) { return kascade_strides{t.stride(0), t.stride(2), t.stride(1)}; }
};

HfTensors hf_tensors(PyObject* const* a) {
    HfTensors h{tensor(a[0], "query"), tensor(a[1], "key"), tensor(a[2], "value")};
    need(h.q.dim() == 4 && h.k.dim() == 4 && h.v.dim() == 4, "query, key and value must be [B,heads,tokens,D]");
    need(h.q.is_cuda() && h.k.is_cuda() && h.v.is_cuda(), "query, key and value must be device tensors");
    h.B = h.q.size(0); h.H = h.q.size(1); h.n = h.q.size(2); h.D = h.q.size(3);
    h.G = h.k.size(1); h.L = h.k.size(2);
    need(h.k.size(0) == h.B && h.k.size(3) == h.D && h.k.sizes() == h.v.sizes() && h.v.scalar_type() == h.k.scalar_type(),
         "key and value must be [B,G,L,D] with query's B and D, of one type");
    h.shape = model_shape(h.q, h.k, h.H, h.G, h.D);
    return h;
}

// Decode reads the head-major cache in place; anything else is brought into [B,tokens,heads,D] order.
void decode_layout(HfTensors& h) {
    need(h.n == 1, "decode takes one query token per sequence");
    if (h.q.stride(3) != 1 || (h.H > 1 && h.q.stride(1) != h.D) || (h.B > 1 && h.q.stride(0) != h.H * h.D)) h.q = h.q.contiguous();
    if (h.k.stride(3) != 1 || h.v.strides() != h.k.strides()) {
        h.k = h.k.transpose(1, 2).contiguous().transpose(1, 2);
        h.v = h.v.transpose(1, 2).contiguous().transpose(1, 2);
    }
}

const at::Tensor& index_lists(PyObject* o, const HfTensors& h) {
    const at::Tensor& idx = dense(o, at::kInt, "topk_indices");
    if (idx.dim() < 3 || idx.size(0) != h.B || idx.size(1) != h.G) fail("index lists must be [%lld,%lld,...,topk]", (long long)h.B, (long long)h.G);
    return idx;
}
const at::Tensor& head_map(PyObject* o, int64_t groups) {
    const at::Tensor& hm = dense(o, at::kInt, "head_mapping");
    if (hm.numel() != groups) fail("head_mapping must have %lld entries", (long long)groups);
    return hm;
}

// Splits of a gather of lists of `topk` rows, and the merge counters it takes (lock held).
struct Gather {
    int64_t topk;
    int ns;
    at::Tensor sync;
};
Gather plan_gather(const HfTensors& h, int64_t topk, PyObject* counters, void* stream) {
    Gather g{topk, 1, {}};
    if (topk > kascade_gather_lone_rows(h.shape.group_size, (int)(h.B * h.G)))
        g.ns = num_split(h.B * h.G, (double)topk, KASCADE_GATHER_ROWS_PER_SPLIT);
    if (g.ns <= KASCADE_FUSED_MERGE_MAX_SPLITS) g.sync = counters_for(counters, stream, h.B * h.G, h.q);
    return g;
}

void hf_reuse(const HfTensors& h, const at::Tensor& idx, const at::Tensor& hm, const Gather& g, const at::Tensor& out,
              void* stream) {
    const int64_t parts = (h.B * h.H * g.ns + 63) / 64 * 64;
    const at::Tensor scratch = empty_like_type({parts + h.B * h.H * g.ns * h.D}, h.q, at::kFloat);
    const kascade_strides st = HfTensors::strides(h.k);
    check(kascade_decode_reuse_paged_shaped_call(
        &h.shape, half_ptr(h.q), half_ptr(h.k), half_ptr(h.v), nullptr, int_ptr(idx), int_ptr(hm), 0.f, float_ptr(scratch),
        float_ptr(scratch) + parts, half_ptr(out), (int)h.B, (int)h.L, (int)g.topk, g.ns, nullptr, 0, 1, &st, nullptr, nullptr,
        g.sync.defined() ? int_ptr(g.sync) : nullptr, nullptr, stream));
}

// hf_decode_reuse(counters, query, key, value, topk_indices, head_mapping) -> O [B,1,H,D]
PyObject* hf_decode_reuse(PyObject* const* a) {
    HfTensors h = hf_tensors(a + 1);
    const at::Tensor& idx = index_lists(a[4], h);
    const at::Tensor& hm = head_map(a[5], h.G);
    void* stream = stream_of(device_of_caller());
    const Gather g = plan_gather(h, idx.size(-1), a[0], stream);
    at::Tensor out;
    {
        Unlocked unlocked;
        decode_layout(h);
        out = at::empty({h.B, 1, h.H, h.D}, h.q.options());
        hf_reuse(h, idx, hm, g, out, stream);
    }
    return THPVariable_Wrap(out);
}

PyObject* pair(const at::Tensor& a, const at::Tensor& b) {
    PyObject* x = THPVariable_Wrap(a);
    PyObject* y = THPVariable_Wrap(b);
    PyObject* t = (x && y) ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    if (!t) throw Fail{};
    return t;
}

// hf_decode_anchor(counters, query, key, value, with_output, width, identity_map) -> (O, topk_indices)
PyObject* hf_decode_anchor(PyObject* const* a) {
    HfTensors h = hf_tensors(a + 1);
    const bool with_output = truth(a[4]);
    const int64_t width = integer(a[5]);
    const at::Tensor& hm = head_map(a[6], h.G);
    need(width > 0, "the selection takes at least one token");
    void* stream = stream_of(device_of_caller());
    const int ns = num_split(h.B * h.G, (double)h.L, 0);
    const int64_t stride = (h.L + 7) / 8 * 8, heads = h.B * h.H;
    auto pad = [](int64_t x) { return (x + 63) / 64 * 64; };
    const int64_t n_lse = pad(heads * ns), n_part = with_output ? pad(heads * ns * h.D) : 0, n_sums = pad(heads);
    Gather g{};
    at::Tensor sync;
    if (!with_output) g = plan_gather(h, width, a[0], stream);
    else if (ns <= KASCADE_FUSED_MERGE_MAX_SPLITS) sync = counters_for(a[0], stream, h.B * h.G, h.q);
    at::Tensor out, idx;
    {
        Unlocked unlocked;
        decode_layout(h);
        const at::Tensor scratch = empty_like_type({n_lse + n_part + n_sums + heads * stride}, h.q, at::kFloat);
        float* lse = float_ptr(scratch);
        float *part = lse + n_lse, *sums = part + n_part, *scores = sums + n_sums;
        const int64_t ws_bytes = kascade_topk_workspace_bytes((int)(h.B * h.G), h.L);
        at::Tensor agg, ws;
        if (h.L > kascade_pool_select_row(h.shape.group_size, (int)(h.B * h.G))) {   // pooled and selected in two launches
            agg = empty_like_type({h.B, h.G, stride}, h.q, at::kHalf);
            if (ws_bytes > 0) ws = empty_like_type({ws_bytes}, h.q, at::kByte);
        }
        out = at::empty({h.B, 1, h.H, h.D}, h.q.options());
        idx = empty_like_type({h.B, h.G, width}, h.q, at::kInt);
        const kascade_strides st = HfTensors::strides(h.k);
        check(kascade_decode_anchor_topk_call(
            &h.shape, half_ptr(h.q), half_ptr(h.k), half_ptr(h.v), nullptr, lse, part, sums, scores,
            with_output ? half_ptr(out) : nullptr, agg.defined() ? half_ptr(agg) : nullptr, int_ptr(idx), nullptr, (int)h.B,
            (int)h.L, (int)stride, ns, with_output, (int)h.L, (int)width, 0, 0.f, nullptr, nullptr,
            ws.defined() ? ws.data_ptr() : nullptr, nullptr, 0, 1, &st, nullptr, nullptr,
            sync.defined() ? int_ptr(sync) : nullptr, stream));
        if (!with_output) hf_reuse(h, idx, hm, g, out, stream);
    }
    return pair(out, idx);
}

// Prompts: strides go to the kernels as they are.
void prompt_layout(const HfTensors& h) {
    need(h.n == h.L, "prefill needs Lq == Lk (no cached prefix), as in the reference kernels");
    need(h.q.stride(3) == 1 && h.k.stride(3) == 1 && h.v.stride(3) == 1, "query, key and value need a contiguous last dimension");
    need(h.v.strides() == h.k.strides(), "K and V must share shape and strides");
}

void prompt_reuse(const HfTensors& h, const at::Tensor& idx, const at::Tensor& hm, float percent, bool rolling,
                  const at::Tensor& out, void* stream) {
    need(idx.dim() == 4 && idx.size(2) == (h.L + 31) / 32, "topk_indices must be [B,G,ceil(L/32),max_topk]");
    check(kascade_prefill_reuse_shaped_call(&h.shape, half_ptr(h.q), half_ptr(h.k), half_ptr(h.v), int_ptr(idx), int_ptr(hm),
                                            percent, half_ptr(out), (int)h.B, (int)h.L, (int)idx.size(3), rolling,
                                            HfTensors::strides(h.q), HfTensors::strides(h.k), nullptr, stream));
}

// hf_prefill_reuse(query, key, value, topk_indices, head_mapping, percent, rolling) -> O [B,L,H,D]
PyObject* hf_prefill_reuse(PyObject* const* a) {
    const HfTensors h = hf_tensors(a);
    prompt_layout(h);
    const at::Tensor& idx = index_lists(a[3], h);
    const at::Tensor& hm = head_map(a[4], h.G);
    const float percent = (float)number(a[5]);
    const bool rolling = truth(a[6]);
    void* stream = stream_of(device_of_caller());
    at::Tensor out;
    {
        Unlocked unlocked;
        out = at::empty({h.B, h.L, h.H, h.D}, h.q.options());
        prompt_reuse(h, idx, hm, percent, rolling, out, stream);
    }
    return THPVariable_Wrap(out);
}

// hf_prefill_anchor(query, key, value, with_output, width, valid_len, n_sel, identity_map, percent, rolling)
// -> (O, topk_indices), for prompts whose pooled scores are formed in one tensor
PyObject* hf_prefill_anchor(PyObject* const* a) {
    const HfTensors h = hf_tensors(a);
    prompt_layout(h);
    const bool with_output = truth(a[3]);
    const int64_t width = integer(a[4]), T = (h.L + 31) / 32;
    const at::Tensor& valid = dense(a[5], at::kInt, "valid_len");
    const at::Tensor& nsel = dense(a[6], at::kInt, "n_sel");
    const at::Tensor& hm = head_map(a[7], h.G);
    need(valid.numel() == T && nsel.numel() == T, "valid_len and n_sel must have one entry per tile");
    const float percent = (float)number(a[8]);
    const bool rolling = truth(a[9]);
    void* stream = stream_of(device_of_caller());
    const kascade_strides qs = HfTensors::strides(h.q), ks = HfTensors::strides(h.k);
    at::Tensor out, idx;
    {
        Unlocked unlocked;
        const at::Tensor log_sum = empty_like_type({h.B, h.L, h.H}, h.q, at::kFloat);
        const at::Tensor scores = empty_like_type({h.B, h.G, T, h.L}, h.q, at::kHalf);
        out = at::empty({h.B, h.L, h.H, h.D}, h.q.options());
        idx = empty_like_type({h.B, h.G, T, width}, h.q, at::kInt);
        check(kascade_prefill_dense_shaped_call(&h.shape, half_ptr(h.q), half_ptr(h.k), with_output ? half_ptr(h.v) : nullptr,
                                                float_ptr(log_sum), with_output ? half_ptr(out) : nullptr, (int)h.B, (int)h.L,
                                                qs, ks, with_output, stream));
        check(kascade_prefill_anchor_topk_call(&h.shape, half_ptr(h.q), half_ptr(h.k), float_ptr(log_sum), half_ptr(scores),
                                               int_ptr(idx), nullptr, (int)h.B, 0, (int)h.L, qs, &ks, nullptr, 0, 1, 0, nullptr,
                                               nullptr, int_ptr(valid), int_ptr(nsel), (int)T, (int)width, (int)h.L - 1, nullptr,
                                               stream));
        if (!with_output) prompt_reuse(h, idx, hm, percent, rolling, out, stream);
    }
    return pair(out, idx);
}

// -------------------------------------------------------------------------- paged cache
// q [B,H,D], pages [P,page,G,D]: any contiguous [...,G,D] view of that memory, where the call does not need
// to know the number of pages
struct PagedTensors {
    at::Tensor q, k, v;
    int64_t B, H, D, G, P, page;
    kascade_shape shape;
};

PagedTensors paged_tensors(PyObject* const* a, long long page, bool counted) {
    PagedTensors t{tensor(a[0], "Q"), tensor(a[1], "K_pages"), tensor(a[2], "V_pages")};
    need(t.q.dim() == 3 && t.k.dim() >= 2 && (t.k.dim() == 4 || !counted), "Q must be [B,H,D] and pages [num_pages,page,G,D]");
    need(t.q.is_cuda() && t.k.is_cuda() && t.v.is_cuda(), "Q, K_pages and V_pages must be device tensors");
    need(t.q.is_contiguous() && t.k.is_contiguous() && t.v.is_contiguous(), "Q, K_pages and V_pages must be contiguous");
    t.B = t.q.size(0); t.H = t.q.size(1); t.D = t.q.size(2);
    t.P = t.k.size(0); t.page = page; t.G = t.k.size(-2);
    t.shape = model_shape(t.q, t.k, t.H, t.G, t.D);
    if ((counted && t.k.size(1) != page) || t.k.size(-1) != t.D || t.k.sizes() != t.v.sizes() || t.v.scalar_type() != t.k.scalar_type())
        fail("pages must be [num_pages,%lld,%lld,%lld]", page, (long long)t.G, (long long)t.D);
    return t;
}

// The caller's output, or none yet.
at::Tensor out_buffer(PyObject* o, const PagedTensors& t) {
    if (o == Py_None) return {};
    const at::Tensor& out = dense(o, t.q.scalar_type(), "out");
    if (out.dim() != 3 || out.size(0) != t.B || out.size(1) != t.H || out.size(2) != t.D)
        fail("out must be [%lld,%lld,%lld]", (long long)t.B, (long long)t.H, (long long)t.D);
    return out;
}

at::Tensor fresh_out(const PagedTensors& t) { return at::empty({t.B, t.H, t.D}, t.q.options()); }

const kascade_half* new_rows(PyObject* o, const PagedTensors& t, const char* name) {
    if (o == Py_None) return nullptr;
    const at::Tensor& r = dense(o, t.q.scalar_type(), name);
    if (r.dim() != 3 || r.size(0) != t.B || r.size(1) != t.G || r.size(2) != t.D)
        fail("%s must be [%lld,%lld,%lld]", name, (long long)t.B, (long long)t.G, (long long)t.D);
    return half_ptr(r);
}

const at::Tensor& table_of(PyObject* o, int64_t B) {
    const at::Tensor& bt = dense(o, at::kInt, "block_table");
    if (bt.dim() != 2 || bt.size(0) != B) fail("block_table must be [%lld,max_pages]", (long long)B);
    return bt;
}
// None: every sequence as long as the call says
const int32_t* lengths_of(PyObject* o, int64_t B) {
    if (o == Py_None) return nullptr;
    const at::Tensor& n = dense(o, at::kInt, "cache_seqlens");
    if (n.numel() != B) fail("cache_seqlens must have %lld entries", (long long)B);
    return int_ptr(n);
}
int32_t* sync_of(PyObject* o, const PagedTensors& t) {
    if (o == Py_None) return nullptr;
    const at::Tensor& s = dense(o, at::kInt, "sync_counters");
    if (s.numel() < t.B * t.G) fail("sync_counters needs %lld entries", (long long)(t.B * t.G));
    return int_ptr(s);
}
void scratch_of(PyObject* lse, PyObject* part, const PagedTensors& t, int64_t ns, float** l, float** p) {
    const at::Tensor& gl = dense(lse, at::kFloat, "glse");
    const at::Tensor& op = dense(part, at::kFloat, "Output_partial");
    if (gl.numel() < t.B * t.H * ns || op.numel() < t.B * t.H * ns * t.D) fail("scratch is too small for %lld splits", (long long)ns);
    *l = float_ptr(gl);
    *p = float_ptr(op);
}

// paged_reuse(Q, K_pages, V_pages, seqlens, cache_rows, head_mapping, percent, glse, Output_partial, num_split,
//             block_table, page_size, out, sync, k_new, v_new) -> O
PyObject* paged_reuse(PyObject* const* a) {
    const PagedTensors t = paged_tensors(a, integer(a[11]), true);
    const int32_t* lens = lengths_of(a[3], t.B);
    const at::Tensor& rows = dense(a[4], at::kInt, "cache_rows");
    if (rows.dim() != 3 || rows.size(0) != t.B || rows.size(1) != t.G) fail("index lists must be [%lld,%lld,topk]", (long long)t.B, (long long)t.G);
    const at::Tensor& hm = head_map(a[5], t.G);
    const int64_t ns = integer(a[9]);
    float *lse, *part;
    scratch_of(a[7], a[8], t, ns, &lse, &part);
    const at::Tensor& bt = table_of(a[10], t.B);
    const float percent = (float)number(a[6]);
    const kascade_half *k_new = new_rows(a[14], t, "k_new"), *v_new = new_rows(a[15], t, "v_new");
    int32_t* sync = sync_of(a[13], t);
    void* stream = stream_of(device_of_caller());
    at::Tensor out = out_buffer(a[12], t);
    {
        Unlocked unlocked;
        if (!out.defined()) out = fresh_out(t);
        check(kascade_decode_reuse_rows_shaped_call(
            &t.shape, half_ptr(t.q), half_ptr(t.k), half_ptr(t.v), lens, int_ptr(rows), int_ptr(hm), percent, lse, part,
            half_ptr(out), (int)t.B, (int)rows.size(2), (int)ns, int_ptr(bt), (int)bt.size(1), (int)t.page, (int)t.P, k_new,
            v_new, sync, nullptr, stream));
    }
    return THPVariable_Wrap(out);
}

// paged_anchor(Q, K_pages, V_pages, seqlens, with_output, glse, Output_partial, num_split, row_sums, scores,
//              max_len, width, percent, valid_len, n_sel, block_table, page_size, out, sync, k_new, v_new, rows_out)
// -> (O or None, topk_indices); cache rows are written to rows_out
PyObject* paged_anchor(PyObject* const* a) {
    const PagedTensors t = paged_tensors(a, integer(a[16]), false);
    const int32_t* lens = lengths_of(a[3], t.B);
    const bool with_output = truth(a[4]);
    const int64_t ns = integer(a[7]), max_len = integer(a[10]), width = integer(a[11]), stride = (max_len + 7) / 8 * 8;
    float *lse, *part;
    scratch_of(a[5], a[6], t, ns, &lse, &part);
    const at::Tensor& sums = dense(a[8], at::kFloat, "row_sums");
    const at::Tensor& scores = dense(a[9], at::kFloat, "scores");
    need(sums.numel() >= t.B * t.H && scores.numel() >= t.B * t.H * stride, "row_sums or scores too small");
    const at::Tensor& bt = table_of(a[15], t.B);
    const at::Tensor& rows = dense(a[21], at::kInt, "rows_out");
    need(rows.numel() >= t.B * t.G * width, "rows_out too small");
    const int32_t *valid = nullptr, *nsel = nullptr;
    if (a[13] != Py_None) {
        const at::Tensor &v = dense(a[13], at::kInt, "valid_len"), &n = dense(a[14], at::kInt, "n_sel");
        need(v.numel() >= t.B * t.G && n.numel() >= t.B * t.G, "valid_len and n_sel need one entry per (sequence, KV head)");
        valid = int_ptr(v);
        nsel = int_ptr(n);
    }
    const float percent = (float)number(a[12]);
    const kascade_half *k_new = new_rows(a[19], t, "k_new"), *v_new = new_rows(a[20], t, "v_new");
    int32_t* sync = sync_of(a[18], t);
    void* stream = stream_of(device_of_caller());
    at::Tensor out, idx, agg, ws;
    if (with_output) out = out_buffer(a[17], t);
    {
        Unlocked unlocked;
        if (with_output && !out.defined()) out = fresh_out(t);
        if (max_len > kascade_pool_select_row(t.shape.group_size, (int)(t.B * t.G))) {
            agg = empty_like_type({t.B, t.G, stride}, t.q, at::kHalf);
            const int64_t bytes = kascade_topk_workspace_bytes((int)(t.B * t.G), max_len);
            if (bytes > 0) ws = empty_like_type({bytes}, t.q, at::kByte);
        }
        idx = empty_like_type({t.B, t.G, width}, t.q, at::kInt);
        check(kascade_decode_anchor_topk_call(
            &t.shape, half_ptr(t.q), half_ptr(t.k), half_ptr(t.v), lens, lse, part, float_ptr(sums), float_ptr(scores),
            with_output ? half_ptr(out) : nullptr, agg.defined() ? half_ptr(agg) : nullptr, int_ptr(idx), int_ptr(rows),
            (int)t.B, (int)max_len, (int)stride, (int)ns, with_output, (int)max_len, (int)width, 0, percent, valid,
            nsel, ws.defined() ? ws.data_ptr() : nullptr, int_ptr(bt), (int)bt.size(1), (int)t.page, nullptr, k_new, v_new, sync,
            stream));
    }
    if (!with_output) {
        PyObject* i = THPVariable_Wrap(idx);
        if (!i) throw Fail{};
        PyObject* r = PyTuple_Pack(2, Py_None, i);
        Py_DECREF(i);
        return r;
    }
    return pair(out, idx);
}

// paged_dense(Q, K_pages, V_pages, seqlens, glse, Output_partial, num_split, max_len, block_table, page_size, out, sync,
//             k_new, v_new) -> O
PyObject* paged_dense(PyObject* const* a) {
    const PagedTensors t = paged_tensors(a, integer(a[9]), false);
    const int32_t* lens = lengths_of(a[3], t.B);
    const int64_t ns = integer(a[6]);
    float *lse, *part;
    scratch_of(a[4], a[5], t, ns, &lse, &part);
    const at::Tensor& bt = table_of(a[8], t.B);
    const int max_len = (int)integer(a[7]);
    const kascade_half *k_new = new_rows(a[12], t, "k_new"), *v_new = new_rows(a[13], t, "v_new");
    int32_t* sync = sync_of(a[11], t);
    void* stream = stream_of(device_of_caller());
    at::Tensor out = out_buffer(a[10], t);
    {
        Unlocked unlocked;
        if (!out.defined()) out = fresh_out(t);
        check(kascade_decode_dense_paged_shaped_call(
            &t.shape, half_ptr(t.q), half_ptr(t.k), half_ptr(t.v), lens, lse, part, half_ptr(out), (int)t.B, max_len, (int)ns,
            int_ptr(bt), (int)bt.size(1), (int)t.page, nullptr, k_new, v_new, sync, stream));
    }
    return THPVariable_Wrap(out);
}

// pool_select_row(group_size, rows): kascade_pool_select_row
PyObject* pool_select_row(PyObject* const* a) {
    return PyLong_FromLong(kascade_pool_select_row((int)integer(a[0]), (int)integer(a[1])));
}

// ------------------------------------------------------------------------------- module
template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
        return nullptr;
    }
    HANDLE_TH_ERRORS   // torch's own errors (out of memory and the like) keep their types
    try {
        return F(args);
    } catch (const Fail&) {
        return nullptr;
    } catch (const Refused& e) {
        PyErr_SetString(g_error, e.message.c_str());
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

#define ENTRY(f, n) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    ENTRY(hf_decode_reuse, 6), ENTRY(hf_decode_anchor, 7), ENTRY(hf_prefill_reuse, 7), ENTRY(hf_prefill_anchor, 10),
    ENTRY(paged_reuse, 16), ENTRY(paged_anchor, 22), ENTRY(paged_dense, 14),
    ENTRY(pool_select_row, 2), {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Per-layer host calls of the Kascade kernels.", -1, kMethods};

PyObject* attribute(const char* module, const char* name) {
    PyObject* m = PyImport_ImportModule(module);
    if (!m) return nullptr;
    PyObject* o = m;
    for (const char* p = name; *p;) {   // dotted path
        const char* dot = strchr(p, '.');
        const std::string part = dot ? std::string(p, dot) : std::string(p);
        PyObject* next = PyObject_GetAttrString(o, part.c_str());
        Py_DECREF(o);
        if (!next) return nullptr;
        o = next;
        p += part.size() + (dot ? 1 : 0);
    }
    return o;
}

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    g_error = attribute("kascade_amd._lib", "KascadeError");
    g_raw_stream = attribute("torch", "_C._cuda_getCurrentRawStream");
    g_capturing = attribute("torch", "_C._cuda_isCurrentStreamCapturing");
    if (!g_error || !g_raw_stream || !g_capturing) return nullptr;
    CountersType.tp_name = "_native.Counters";
    CountersType.tp_basicsize = sizeof(Counters);
    CountersType.tp_flags = Py_TPFLAGS_DEFAULT;
    CountersType.tp_new = counters_new;
    CountersType.tp_dealloc = counters_dealloc;
    if (PyType_Ready(&CountersType) < 0) return nullptr;
    PyObject* m = PyModule_Create(&kModule);
    if (!m) return nullptr;
    Py_INCREF(&CountersType);
    if (PyModule_AddObject(m, "Counters", reinterpret_cast<PyObject*>(&CountersType)) < 0) return nullptr;
    return m;
}
