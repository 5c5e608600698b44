// extern "C" entry points of libkascade_hip.so: argument validation, launch
// sequencing, error reporting.  No allocation happens here; every buffer is the
// caller's.  Validation failures are reported before anything is launched, so
// they can be exercised on a machine without a GPU.
#include "../../include/kascade_hip.h"
#include "../../include/kascade_hip_diag.h"

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <mutex>

#include "decode.h"
#include "diag.h"
#include "paged.h"
#include "prefill.h"
#include "topk.h"

using namespace kascade;

namespace {

thread_local char g_err[1024] = "";
int g_cu_count = 0;

// Scratch of kascade_decode_reuse_paged_noalloc_call: the partial log-sums [batch,32,num_split]
// and partial outputs [batch,32,num_split,128] of the splits, fp32, for up to kNoAllocUnits
// (sequence, split) pairs.  Every device the library runs on holds its own copy of the array at
// its own address until the process ends; host code never uses the array's name as an address but
// the pointer hipGetSymbolAddress returns for the current device (g_noalloc_ptr).
constexpr int kNoAllocUnits = 1024;
constexpr size_t kNoAllocFloats = (size_t)kNoAllocUnits * kHeads * (1 + kDim);   // 16.9 MB
static __device__ __align__(256) float scratch[kNoAllocFloats];
constexpr int kMaxDevices = 64;
float* g_noalloc_ptr[kMaxDevices] = {};
std::mutex g_noalloc_mutex;   // host threads that meet in the first call on a device

int fail(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return -1;
}

int check_hip(hipError_t e, const char* what) {
    if (e == hipSuccess) return 0;
    return fail("%s: %s", what, hipGetErrorString(e));
}

#define REQUIRE(cond, ...)                 \
    do {                                   \
        if (!(cond)) return fail(__VA_ARGS__); \
    } while (0)

inline const half_t* H(const kascade_half* p) { return reinterpret_cast<const half_t*>(p); }
inline half_t* H(kascade_half* p) { return reinterpret_cast<half_t*>(p); }
// element tensors whose type (fp16 or bf16) the shape decides
inline const void* E(const kascade_half* p) { return p; }
inline void* E(kascade_half* p) { return p; }

// Device address of `scratch` on the current device, looked up once per device.
int noalloc_scratch(float** out) {
    int dev = 0;
    if (check_hip(hipGetDevice(&dev), "hipGetDevice")) return -1;
    REQUIRE(dev >= 0 && dev < kMaxDevices, "device ordinal %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_noalloc_mutex);
    if (!g_noalloc_ptr[dev]) {
        void* ptr = nullptr;
        if (check_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)"))
            return -1;
        REQUIRE(ptr != nullptr, "hipGetSymbolAddress(scratch) returned a null address");
        g_noalloc_ptr[dev] = static_cast<float*>(ptr);
    }
    *out = g_noalloc_ptr[dev];
    return 0;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int check_strides(const kascade_strides& s, const char* name) {
    REQUIRE(s.b % 8 == 0 && s.l % 8 == 0 && s.h % 8 == 0,
            "%s strides must be multiples of 8 elements (16-byte rows)", name);
    REQUIRE(s.l > 0 && s.h > 0, "%s strides must be positive", name);
    REQUIRE(s.l < (1LL << 31), "%s row stride must be below 2^31 elements", name);
    return 0;
}

// Shape of the tensors a call works on: KV heads, head dimension, element kind, query heads per
// KV head.  The entry points without a shape argument use the reference's.
struct Shape {
    int G, D, elem, gs;
    int H() const { return G * gs; }
};
const Shape kRefShape{kGroups, kDim, kElemF16, kGroupSize};

int get_shape(const kascade_shape* in, Shape* out) {
    REQUIRE(in, "shape: null pointer argument");
    REQUIRE(in->kv_heads >= 1 && in->kv_heads <= 65535, "shape: kv_heads out of range");
    REQUIRE(in->head_dim == 64 || in->head_dim == 128, "shape: head_dim must be 64 or 128, got %d", in->head_dim);
    REQUIRE(in->dtype == KASCADE_F16 || in->dtype == KASCADE_BF16, "shape: dtype must be KASCADE_F16 or KASCADE_BF16");
    const int gs = in->group_size == 0 ? kGroupSize : in->group_size;
    REQUIRE(gs >= 1 && gs <= 16,
            "shape: group_size (query heads per KV head) must be 1 to 16 (0 = 4), got %d", in->group_size);
    REQUIRE((long long)in->kv_heads * gs <= 65535, "shape: too many query heads");
    out->G = in->kv_heads; out->D = in->head_dim; out->elem = in->dtype == KASCADE_BF16 ? kElemBF16 : kElemF16;
    out->gs = gs;
    return 0;
}

// what the reference's scratch shapes fix for its decode kernels (attention_utils.py:36-59)
constexpr int kRefNumSplit = 8;

// element strides of a contiguous [B,seq_len,heads,128] tensor
kascade_strides contiguous_strides(int seq_len, int heads) {
    return kascade_strides{(int64_t)seq_len * heads * kDim, (int64_t)heads * kDim, (int64_t)kDim};
}

int rows_per_split(long long max_rows, int num_split) {
    long long r = (max_rows + num_split - 1) / num_split;
    return (int)(((r + 63) / 64) * 64);
}

int check_paging(const int32_t* block_table, int max_pages, int page_size, int* page_shift) {
    if (!block_table) {
        *page_shift = 0;
        return 0;
    }
    int sh = ilog2_exact(page_size);
    REQUIRE(sh >= 0, "page_size must be a power of two, got %d", page_size);
    REQUIRE(max_pages > 0, "max_pages must be positive with a block table");
    *page_shift = sh;
    return 0;
}

// K/V addressing of the decode calls without a block table: `strides` (elements, may be NULL
// for the contiguous [B,kv_stride_tokens,G,D] cache).
int set_kv_strides(DecodeParams& p, const Shape& sh, const kascade_strides* strides,
                   const int32_t* block_table, int kv_stride_tokens) {
    p.G = sh.G; p.head_dim = sh.D; p.elem = sh.elem; p.gs = sh.gs;
    if (!strides) {
        p.kv_stride_b = (long long)kv_stride_tokens * sh.G * sh.D;
        p.kv_stride_l = sh.G * sh.D;
        p.kv_stride_h = sh.D;
        return 0;
    }
    REQUIRE(!block_table, "kv_strides and block_table exclude each other");
    if (check_strides(*strides, "decode K/V")) return -1;
    REQUIRE(strides->b >= 0, "decode K/V batch stride must not be negative");
    p.kv_stride_b = strides->b;
    p.kv_stride_l = (unsigned)strides->l;
    p.kv_stride_h = strides->h;
    return 0;
}

// Fused append of the decode calls: both rows or neither; the caches are written through the
// K / V arguments.
int set_append(DecodeParams& p, const kascade_half* k_new, const kascade_half* v_new,
               const kascade_half* K, const kascade_half* V) {
    if (!k_new && !v_new) return 0;
    REQUIRE(k_new && v_new && K && V, "k_new and v_new come together, with both caches");
    REQUIRE(aligned16(k_new) && aligned16(v_new), "k_new/v_new must be 16-byte aligned");
    p.k_new = H(k_new); p.v_new = H(v_new);
    p.k_cache = const_cast<half_t*>(H(K)); p.v_cache = const_cast<half_t*>(H(V));
    return 0;
}

}  // namespace

extern "C" {

int kascade_abi_version(void) { return 13; }

const char* kascade_get_last_error(void) { return g_err; }

int kascade_device_cu_count(void) { return g_cu_count; }

int kascade_init(void) {
    int dev = 0;
    if (check_hip(hipGetDevice(&dev), "hipGetDevice")) return -1;
    hipDeviceProp_t prop;
    if (check_hip(hipGetDeviceProperties(&prop, dev), "hipGetDeviceProperties")) return -1;
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail("libkascade_hip is built for gfx950 only; device is %s", prop.gcnArchName);
    g_cu_count = prop.multiProcessorCount;
    float* ptr;
    return noalloc_scratch(&ptr);   // this device's copy of the scratch array
}

int kascade_decode_reuse_call(const kascade_half* Q, const kascade_half* K, const kascade_half* V,
                              const int32_t* topk_indices, const int32_t* head_mapping,
                              float* glse, float* Output_partial, kascade_half* Output, int batch,
                              int kv_seqlen, int topk, int num_split, int32_t* sync_counters,
                              void* stream) {
    return kascade_decode_reuse_paged_call(Q, K, V, nullptr, topk_indices, head_mapping, 0.f, glse,
                                           Output_partial, Output, batch, kv_seqlen, topk,
                                           num_split, nullptr, 0, 1, nullptr, nullptr, nullptr, sync_counters,
                                           nullptr, stream);
}

}  // extern "C"
namespace {
int decode_reuse_paged_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K,
                                    const kascade_half* V, const int32_t* cache_seqlens,
                                    const int32_t* topk_indices, const int32_t* head_mapping,
                                    float topk_percent, float* glse, float* Output_partial,
                                    kascade_half* Output, int batch, int kv_stride_tokens,
                                    int topk, int num_split, const int32_t* block_table,
                                    int max_pages, int page_size, const kascade_strides* kv_strides,
                                    const kascade_half* k_new, const kascade_half* v_new,
                                    int32_t* sync_counters, float* log_sum, void* stream) {
    REQUIRE(Q && K && V && topk_indices && head_mapping && glse && Output_partial && Output,
            "decode_reuse: null pointer argument");
    REQUIRE(batch > 0 && topk > 0 && num_split > 0, "decode_reuse: batch, topk, num_split must be > 0");
    REQUIRE(batch <= 65535, "decode_reuse: batch exceeds grid limit");
    REQUIRE(block_table || kv_stride_tokens > 0, "decode_reuse: kv_stride_tokens must be > 0");
    REQUIRE(!(topk_percent > 0.f) || cache_seqlens, "decode_reuse: topk_percent needs cache_seqlens");
    REQUIRE(aligned16(Q) && aligned16(K) && aligned16(V), "decode_reuse: Q/K/V must be 16-byte aligned");
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    DecodeParams p{};
    p.Q = H(Q); p.K = H(K); p.V = H(V);
    p.seqlens = cache_seqlens; p.idx = topk_indices; p.head_map = head_mapping;
    p.block_table = block_table; p.glse = glse; p.opart = Output_partial; p.scores = nullptr;
    p.max_pages = max_pages; p.page_shift = shift; p.kv_stride_tokens = kv_stride_tokens;
    if (set_kv_strides(p, sh, kv_strides, block_table, kv_stride_tokens)) return -1;
    if (set_append(p, k_new, v_new, K, V)) return -1;
    p.topk = topk; p.topk_percent = topk_percent; p.scores_stride = 0; p.num_split = num_split;
    p.rows_per_split = rows_per_split(topk, num_split);
    p.B = batch;
    p.counters = sync_counters; p.out = H(Output); p.row_sums = log_sum;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (check_hip(launch_decode_split(p, true, true, false, s), "decode_reuse split")) return -1;
    if (sync_counters) return 0;   // the split kernel's last workgroups have combined
    return check_hip(launch_decode_combine(glse, Output_partial, E(Output), log_sum, batch, sh.H(), num_split, true, sh.D, sh.elem, s), "decode_reuse combine");
}
}  // namespace
extern "C" {

int kascade_decode_reuse_paged_call(const kascade_half* Q, const kascade_half* K,
                                    const kascade_half* V, const int32_t* cache_seqlens,
                                    const int32_t* topk_indices, const int32_t* head_mapping,
                                    float topk_percent, float* glse, float* Output_partial,
                                    kascade_half* Output, int batch, int kv_stride_tokens,
                                    int topk, int num_split, const int32_t* block_table,
                                    int max_pages, int page_size, const kascade_strides* kv_strides,
                                    const kascade_half* k_new, const kascade_half* v_new,
                                    int32_t* sync_counters, float* log_sum, void* stream) {
    return decode_reuse_paged_impl(kRefShape, Q, K, V, cache_seqlens, topk_indices, head_mapping, topk_percent, glse, Output_partial, Output, batch, kv_stride_tokens, topk, num_split, block_table, max_pages, page_size, kv_strides, k_new, v_new, sync_counters, log_sum, stream);
}

int kascade_decode_reuse_paged_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K,
                                    const kascade_half* V, const int32_t* cache_seqlens,
                                    const int32_t* topk_indices, const int32_t* head_mapping,
                                    float topk_percent, float* glse, float* Output_partial,
                                    kascade_half* Output, int batch, int kv_stride_tokens,
                                    int topk, int num_split, const int32_t* block_table,
                                    int max_pages, int page_size, const kascade_strides* kv_strides,
                                    const kascade_half* k_new, const kascade_half* v_new,
                                    int32_t* sync_counters, float* log_sum, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return decode_reuse_paged_impl(sh, Q, K, V, cache_seqlens, topk_indices, head_mapping, topk_percent, glse, Output_partial, Output, batch, kv_stride_tokens, topk, num_split, block_table, max_pages, page_size, kv_strides, k_new, v_new, sync_counters, log_sum, stream);
}

}  // extern "C"
namespace {
int decode_reuse_rows_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K_pages,
                                   const kascade_half* V_pages, const int32_t* cache_seqlens,
                                   const int32_t* cache_rows, const int32_t* head_mapping,
                                   float topk_percent, float* glse, float* Output_partial,
                                   kascade_half* Output, int batch, int topk, int num_split,
                                   const int32_t* block_table, int max_pages, int page_size,
                                   int num_pages, const kascade_half* k_new,
                                   const kascade_half* v_new, int32_t* sync_counters, float* log_sum, void* stream) {
    REQUIRE(Q && K_pages && V_pages && cache_rows && head_mapping && glse && Output_partial && Output &&
                block_table, "decode_reuse_rows: null pointer argument");
    REQUIRE(batch > 0 && topk > 0 && num_split > 0, "decode_reuse_rows: batch, topk, num_split must be > 0");
    REQUIRE(batch <= 65535, "decode_reuse_rows: batch exceeds grid limit");
    REQUIRE(!(topk_percent > 0.f) || cache_seqlens, "decode_reuse_rows: topk_percent needs cache_seqlens");
    REQUIRE(!k_new || cache_seqlens, "decode_reuse_rows: the fused append needs cache_seqlens");
    REQUIRE(aligned16(Q) && aligned16(K_pages) && aligned16(V_pages),
            "decode_reuse_rows: Q/K/V must be 16-byte aligned");
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    REQUIRE(num_pages > 0 && (long long)num_pages * page_size < (1LL << 31),
            "decode_reuse_rows: num_pages out of range");
    DecodeParams p{};
    p.Q = H(Q); p.K = H(K_pages); p.V = H(V_pages);
    p.seqlens = cache_seqlens; p.idx = cache_rows; p.head_map = head_mapping;
    p.idx_physical = 1; p.max_row = num_pages * page_size - 1;
    p.block_table = block_table; p.glse = glse; p.opart = Output_partial; p.scores = nullptr;
    p.max_pages = max_pages; p.page_shift = shift; p.kv_stride_tokens = 0;
    if (set_kv_strides(p, sh, nullptr, block_table, 0)) return -1;
    if (set_append(p, k_new, v_new, K_pages, V_pages)) return -1;
    p.topk = topk; p.topk_percent = topk_percent; p.scores_stride = 0; p.num_split = num_split;
    p.rows_per_split = rows_per_split(topk, num_split);
    p.B = batch;
    p.counters = sync_counters; p.out = H(Output); p.row_sums = log_sum;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (check_hip(launch_decode_split(p, true, true, false, s), "decode_reuse_rows split")) return -1;
    if (sync_counters) return 0;
    return check_hip(launch_decode_combine(glse, Output_partial, E(Output), log_sum, batch, sh.H(), num_split, true, sh.D, sh.elem, s), "decode_reuse_rows combine");
}
}  // namespace
extern "C" {

int kascade_decode_reuse_rows_call(const kascade_half* Q, const kascade_half* K_pages,
                                   const kascade_half* V_pages, const int32_t* cache_seqlens,
                                   const int32_t* cache_rows, const int32_t* head_mapping,
                                   float topk_percent, float* glse, float* Output_partial,
                                   kascade_half* Output, int batch, int topk, int num_split,
                                   const int32_t* block_table, int max_pages, int page_size,
                                   int num_pages, const kascade_half* k_new,
                                   const kascade_half* v_new, int32_t* sync_counters, float* log_sum, void* stream) {
    return decode_reuse_rows_impl(kRefShape, Q, K_pages, V_pages, cache_seqlens, cache_rows, head_mapping, topk_percent, glse, Output_partial, Output, batch, topk, num_split, block_table, max_pages, page_size, num_pages, k_new, v_new, sync_counters, log_sum, stream);
}

int kascade_decode_reuse_rows_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K_pages,
                                   const kascade_half* V_pages, const int32_t* cache_seqlens,
                                   const int32_t* cache_rows, const int32_t* head_mapping,
                                   float topk_percent, float* glse, float* Output_partial,
                                   kascade_half* Output, int batch, int topk, int num_split,
                                   const int32_t* block_table, int max_pages, int page_size,
                                   int num_pages, const kascade_half* k_new,
                                   const kascade_half* v_new, int32_t* sync_counters, float* log_sum, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return decode_reuse_rows_impl(sh, Q, K_pages, V_pages, cache_seqlens, cache_rows, head_mapping, topk_percent, glse, Output_partial, Output, batch, topk, num_split, block_table, max_pages, page_size, num_pages, k_new, v_new, sync_counters, log_sum, stream);
}

int kascade_decode_reuse_paged_noalloc_call(const kascade_half* Q, const kascade_half* K,
                                            const kascade_half* V, const int32_t* cache_seqlens,
                                            const int32_t* topk_indices, const int32_t* head_mapping,
                                            float topk_percent, kascade_half* Output, int batch,
                                            int kv_stride_tokens, int topk, int num_split,
                                            const int32_t* block_table, int max_pages, int page_size,
                                            const kascade_strides* kv_strides,
                                            const kascade_half* k_new, const kascade_half* v_new,
                                            void* stream) {
    REQUIRE(batch > 0 && num_split > 0, "decode_reuse_noalloc: batch, num_split must be > 0");
    REQUIRE((long long)batch * num_split <= kNoAllocUnits,
            "decode_reuse_noalloc: batch * num_split = %lld exceeds the built-in scratch (%d); "
            "use kascade_decode_reuse_paged_call with caller-provided scratch",
            (long long)batch * num_split, kNoAllocUnits);
    float* base;
    if (noalloc_scratch(&base)) return -1;
    float* glse = base;                                           // [batch,32,num_split]
    float* opart = base + (size_t)kNoAllocUnits * kHeads;         // [batch,32,num_split,128]
    return decode_reuse_paged_impl(kRefShape, Q, K, V, cache_seqlens, topk_indices, head_mapping,
                                           topk_percent, glse, opart, Output, batch,
                                           kv_stride_tokens, topk, num_split, block_table, max_pages,
                                           page_size, kv_strides, k_new, v_new, nullptr, nullptr, stream);
}

}  // extern "C"
namespace {
int decode_dense_paged_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K,
                                    const kascade_half* V, const int32_t* cache_seqlens,
                                    float* glse, float* Output_partial, kascade_half* Output,
                                    int batch, int kv_stride_tokens, int num_split,
                                    const int32_t* block_table, int max_pages, int page_size,
                                    const kascade_strides* kv_strides, const kascade_half* k_new,
                                    const kascade_half* v_new, int32_t* sync_counters,
                                    void* stream) {
    REQUIRE(Q && K && V && glse && Output_partial && Output, "decode_dense: null pointer argument");
    REQUIRE(batch > 0 && num_split > 0, "decode_dense: batch, num_split must be > 0");
    REQUIRE(batch <= 65535, "decode_dense: batch exceeds grid limit");
    REQUIRE(cache_seqlens || kv_stride_tokens > 0, "decode_dense: need cache_seqlens or kv_stride_tokens");
    REQUIRE(block_table || kv_stride_tokens > 0, "decode_dense: kv_stride_tokens must be > 0");
    REQUIRE(aligned16(Q) && aligned16(K) && aligned16(V), "decode_dense: Q/K/V must be 16-byte aligned");
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    DecodeParams p{};
    p.Q = H(Q); p.K = H(K); p.V = H(V);
    p.seqlens = cache_seqlens; p.block_table = block_table; p.glse = glse; p.opart = Output_partial;
    p.max_pages = max_pages; p.page_shift = shift; p.kv_stride_tokens = kv_stride_tokens;
    if (set_kv_strides(p, sh, kv_strides, block_table, kv_stride_tokens)) return -1;
    if (set_append(p, k_new, v_new, K, V)) return -1;
    p.num_split = num_split; p.B = batch;
    const long long max_rows = kv_stride_tokens > 0 ? kv_stride_tokens : (long long)max_pages * page_size;
    p.rows_per_split = rows_per_split(max_rows, num_split);
    p.counters = sync_counters; p.out = H(Output);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (check_hip(launch_decode_split(p, false, true, false, s), "decode_dense split")) return -1;
    if (sync_counters) return 0;
    return check_hip(launch_decode_combine(glse, Output_partial, E(Output), nullptr, batch, sh.H(), num_split, true, sh.D, sh.elem, s), "decode_dense combine");
}
}  // namespace
extern "C" {

int kascade_decode_dense_paged_call(const kascade_half* Q, const kascade_half* K,
                                    const kascade_half* V, const int32_t* cache_seqlens,
                                    float* glse, float* Output_partial, kascade_half* Output,
                                    int batch, int kv_stride_tokens, int num_split,
                                    const int32_t* block_table, int max_pages, int page_size,
                                    const kascade_strides* kv_strides, const kascade_half* k_new,
                                    const kascade_half* v_new, int32_t* sync_counters,
                                    void* stream) {
    return decode_dense_paged_impl(kRefShape, Q, K, V, cache_seqlens, glse, Output_partial, Output, batch, kv_stride_tokens, num_split, block_table, max_pages, page_size, kv_strides, k_new, v_new, sync_counters, stream);
}

int kascade_decode_dense_paged_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K,
                                    const kascade_half* V, const int32_t* cache_seqlens,
                                    float* glse, float* Output_partial, kascade_half* Output,
                                    int batch, int kv_stride_tokens, int num_split,
                                    const int32_t* block_table, int max_pages, int page_size,
                                    const kascade_strides* kv_strides, const kascade_half* k_new,
                                    const kascade_half* v_new, int32_t* sync_counters,
                                    void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return decode_dense_paged_impl(sh, Q, K, V, cache_seqlens, glse, Output_partial, Output, batch, kv_stride_tokens, num_split, block_table, max_pages, page_size, kv_strides, k_new, v_new, sync_counters, stream);
}

}  // extern "C"
namespace {
// The selection that follows an anchor pass in the same call.
struct AnchorSelect {
    bool one_launch;           // pooling and selection together
    int32_t* out_idx;
    const TopkRows* rows;      // or null
    int row_len, k, fill;
    float topk_percent;
    const int32_t *valid_len, *n_sel;   // long rows only
    void* workspace;
};

static_assert(KASCADE_POOL_SELECT_ROW == kPoolSelectRow, "the header's limit is the kernel's");

// rows that start 16-byte aligned and fit one workgroup's registers
bool one_workgroup_rows(int len) { return len <= topk_max_register_row(); }

// Selection over a tensor of scores, as kascade_topk_rows_call describes it (arguments checked).
int select_rows(const half_t* scores, int32_t* out_idx, int rows, int64_t row_stride, int uniform_len,
                const int32_t* valid_len, const int32_t* n_sel, int period, int k, int fill_value,
                void* workspace, const TopkRows& tr, hipStream_t s) {
    // rows of up to 131072 entries fit one workgroup's registers: one launch; longer (or unaligned
    // long) rows go to several workgroups per row, four launches
    const bool one_workgroup = one_workgroup_rows(uniform_len + (row_stride % 8 != 0 ? 7 : 0)) &&
                               (reinterpret_cast<uintptr_t>(scores) & 15) == 0;
    if (!one_workgroup && workspace && topk_split_workspace_bytes(rows, uniform_len) > 0)
        return check_hip(launch_topk_split(scores, out_idx, rows, row_stride, uniform_len,
                                           uniform_len, valid_len, n_sel, period, k, fill_value,
                                           workspace, &tr, s), "topk (split)");
    return check_hip(launch_topk(scores, out_idx, rows, row_stride, uniform_len, valid_len, n_sel,
                                 period, k, fill_value, &tr, s), "topk");
}

int decode_recompute_paged_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K,
                                        const kascade_half* V, const int32_t* cache_seqlens,
                                        float* glse, float* Output_partial, float* row_sums,
                                        float* scores, kascade_half* Output,
                                        kascade_half* aggregated_scores, int batch,
                                        int kv_stride_tokens, int scores_stride, int num_split,
                                        int with_output, const int32_t* block_table,
                                        int max_pages, int page_size,
                                        const kascade_strides* kv_strides,
                                        const kascade_half* k_new, const kascade_half* v_new,
                                        int32_t* sync_counters, const AnchorSelect* sel, void* stream) {
    REQUIRE(Q && K && glse && row_sums && scores && (aggregated_scores || (sel && sel->one_launch)),
            "decode_recompute: null pointer argument");
    REQUIRE(!with_output || (V && Output && Output_partial),
            "decode_recompute: with_output needs V, Output and Output_partial");
    REQUIRE(batch > 0 && num_split > 0 && scores_stride > 0,
            "decode_recompute: batch, num_split, scores_stride must be > 0");
    REQUIRE(scores_stride % 8 == 0, "decode_recompute: scores_stride must be a multiple of 8");
    REQUIRE(batch <= 65535, "decode_recompute: batch exceeds grid limit");
    REQUIRE(cache_seqlens || (kv_stride_tokens > 0 && kv_stride_tokens <= scores_stride),
            "decode_recompute: without cache_seqlens need 0 < kv_stride_tokens <= scores_stride");
    REQUIRE(block_table || kv_stride_tokens > 0, "decode_recompute: kv_stride_tokens must be > 0");
    REQUIRE(aligned16(Q) && aligned16(K) && (!with_output || aligned16(V)),
            "decode_recompute: Q/K/V must be 16-byte aligned");
    REQUIRE(aligned16(scores) && aligned16(aggregated_scores),
            "decode_recompute: scores buffers must be 16-byte aligned");
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    DecodeParams p{};
    p.Q = H(Q); p.K = H(K); p.V = with_output ? H(V) : H(K);
    p.seqlens = cache_seqlens; p.block_table = block_table; p.glse = glse; p.opart = Output_partial;
    p.scores = scores; p.scores_stride = scores_stride;
    p.max_pages = max_pages; p.page_shift = shift; p.kv_stride_tokens = kv_stride_tokens;
    if (set_kv_strides(p, sh, kv_strides, block_table, kv_stride_tokens)) return -1;
    if (set_append(p, k_new, v_new, K, V)) return -1;
    p.num_split = num_split; p.B = batch;
    long long max_rows = kv_stride_tokens > 0 ? kv_stride_tokens : (long long)max_pages * page_size;
    if (max_rows > scores_stride) max_rows = scores_stride;
    p.rows_per_split = rows_per_split(max_rows, num_split);
    p.counters = sync_counters; p.out = H(Output); p.row_sums = row_sums;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // Without an output the only thing left to merge is the log-sums, which the pooling launch does
    // for itself: no combine launch, no counters.
    if (!with_output) p.counters = nullptr;
    if (check_hip(launch_decode_split(p, false, with_output != 0, true, s), "decode_recompute split"))
        return -1;
    // the kernels cut every sequence length down to this (decode_split_kernel's safe_len)
    long long len_cap = block_table ? (long long)max_pages * page_size : (long long)kv_stride_tokens;
    if (len_cap > scores_stride) len_cap = scores_stride;
    if (!sync_counters && with_output &&
        check_hip(launch_decode_combine(glse, Output_partial, E(Output), row_sums, batch, sh.H(), num_split, true, sh.D, sh.elem, s), "decode_recompute combine"))
        return -1;
    const float* parts = with_output ? nullptr : glse;   // log-sums still to be merged
    const TopkRows no_rows{};
    if (sel && sel->one_launch) {
        DecodePoolParams pp{};
        pp.scores = scores; pp.glse = parts; pp.row_sums = row_sums; pp.seqlens = cache_seqlens;
        pp.num_split = num_split; pp.groups = sh.G; pp.group_size = sh.gs; pp.scores_stride = scores_stride;
        pp.uniform_len = sel->row_len; pp.len_cap = (int)len_cap; pp.topk_percent = sel->topk_percent;
        return check_hip(launch_decode_pool_select(pp, batch * sh.G, sel->k, sel->fill, sel->out_idx,
                                                   sel->rows ? sel->rows : &no_rows, s), "decode_anchor pool+topk");
    }
    if (check_hip(launch_decode_aggregate(scores, with_output ? row_sums : nullptr, parts, num_split, row_sums,
                                          cache_seqlens, H(aggregated_scores), batch, sh.G, sh.gs, scores_stride,
                                          kv_stride_tokens, (int)len_cap, s),
                  "decode_recompute aggregate"))
        return -1;
    if (!sel) return 0;
    return select_rows(H(aggregated_scores), sel->out_idx, batch * sh.G, scores_stride, sel->row_len, sel->valid_len,
                       sel->n_sel, batch * sh.G, sel->k, sel->fill, sel->workspace, sel->rows ? *sel->rows : no_rows, s);
}
}  // namespace
extern "C" {

int kascade_decode_recompute_paged_call(const kascade_half* Q, const kascade_half* K,
                                        const kascade_half* V, const int32_t* cache_seqlens,
                                        float* glse, float* Output_partial, float* row_sums,
                                        float* scores, kascade_half* Output,
                                        kascade_half* aggregated_scores, int batch,
                                        int kv_stride_tokens, int scores_stride, int num_split,
                                        int with_output, const int32_t* block_table,
                                        int max_pages, int page_size,
                                        const kascade_strides* kv_strides,
                                        const kascade_half* k_new, const kascade_half* v_new,
                                        int32_t* sync_counters, void* stream) {
    return decode_recompute_paged_impl(kRefShape, Q, K, V, cache_seqlens, glse, Output_partial, row_sums, scores, Output, aggregated_scores, batch, kv_stride_tokens, scores_stride, num_split, with_output, block_table, max_pages, page_size, kv_strides, k_new, v_new, sync_counters, nullptr, stream);
}

int kascade_decode_recompute_paged_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K,
                                        const kascade_half* V, const int32_t* cache_seqlens,
                                        float* glse, float* Output_partial, float* row_sums,
                                        float* scores, kascade_half* Output,
                                        kascade_half* aggregated_scores, int batch,
                                        int kv_stride_tokens, int scores_stride, int num_split,
                                        int with_output, const int32_t* block_table,
                                        int max_pages, int page_size,
                                        const kascade_strides* kv_strides,
                                        const kascade_half* k_new, const kascade_half* v_new,
                                        int32_t* sync_counters, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return decode_recompute_paged_impl(sh, Q, K, V, cache_seqlens, glse, Output_partial, row_sums, scores, Output, aggregated_scores, batch, kv_stride_tokens, scores_stride, num_split, with_output, block_table, max_pages, page_size, kv_strides, k_new, v_new, sync_counters, nullptr, stream);
}

int kascade_decode_num_split(double total_rows, double max_rows, int compute_units, double wgs_per_cu, double min_rows,
                             double cap_rows) {
    double per = fmax(min_rows, total_rows / (wgs_per_cu * compute_units));
    if (cap_rows > 0) per = fmin(per, cap_rows);
    // small launch (short lists, small batch): latency, not set-up, is what counts, so spread down to
    // 128 rows per workgroup to put one workgroup on every compute unit
    const bool small = total_rows / per < compute_units;
    if (small) per = fmax(fmin(128, min_rows), total_rows / compute_units);
    if (per <= 0) return 1;
    double ns = fmax(1, fmin(256, nearbyint(max_rows / per)));
    // Small gathers stop at 64 splits, or what cap_rows asks for, whatever part of max_rows is filled.  Us, batch 1, 32/8 heads,
    // room for 13184 rows, with 64 / 103 splits (128 rows each): 512 rows 10.3/10.8, 1664 10.9/11.5, 3328 11.6/12.3, 6656
    // 13.0/15.6, 13184 18.8/24.8; 12032 rows at 8/2 heads of 64 with 64 / 94: 10.7/12.7.
    if (small && cap_rows > 0) ns = fmin(ns, fmax(64, ceil(max_rows / cap_rows)));
    // to the nearest: one workgroup more than a whole number per compute unit costs a full extra wave
    // of workgroups on a few units, one fewer costs nothing
    return (int)ns;
}

}  // extern "C"
namespace {
// Splits per list that make whole rounds of workgroups: one on (almost) every unit, or two where those fill the chip better by
// more than an eighth.  A gather whose splits would in one round be longer than cap_rows, and than num_split makes them, takes
// two, or three on the same terms (8 KV heads, 22 sequences' lists of 6656 rows, us by splits: 2 124, 3 127, 4 107; 17: 3
// 88.2, 4 94.5, 5 85.3; 25: 2 130, 3 135, 4 134).
int whole_rounds(int lists, double rows, int num_split, int compute_units, double cap_rows) {
    const auto splits = [&](int rounds) { return fmax(1, floor((double)rounds * compute_units / lists)); };
    const auto fill = [&](int rounds) { return splits(rounds) * lists / ((double)rounds * compute_units); };
    const bool too_long = cap_rows > 0 && rows / splits(1) > fmax(cap_rows, rows / num_split);
    int rounds = lists <= compute_units && !too_long && fill(1) >= fill(2) - 0.125 ? 1 : 2;
    if (too_long && fill(3) > fill(2) + 0.125) rounds = 3;
    return (int)fmin(256, splits(rounds));
}
}  // namespace
extern "C" {

// Lists of different lengths fill in behind each other (a gather of 17 sequences' lists of 512 to 896 rows by this rule: its
// step 1.5 % slower); equal ones do not.  Between one workgroup per compute unit and two, the units with two finish last
// and the others wait.  Us per launch (anchor pass with output / without, pooling launch included; gathers of 10 %) by
// splits, the nearest count first:
//   8 x 3000 tokens, 64/8 heads    6: 37.7/35.3   4: 34.3/33.2   8: 35.7/34.4
//   2 x 9000, 64/8                18: 41.9/39.6  16: 37.0/37.2  32: 39.2/37.7
//   9 x 2500, 32/8                 5: 35.5/31.4   3: 31.9/29.2   7: 31.5/29.1
//   12 x 1200, 32/8                3: 28.7/25.5   2: 25.7/23.8   5: 24.3/23.0
//   36 x 5000, 8/2 heads of 64     4: 37.2/36.2   3: 35.5/34.8   7: 32.4/31.9
//   gather of 12 x 896 rows        3: 17.7        2: 15.1        5: 15.4
//   gather of 9 x 1664 rows        4: 22.4        3: 18.3        7: 17.3
//   gather of 7 x 1664, 64/8       5: 21.1        4: 16.9        9: 17.7
// and with many lists, where one round leaves up to a third of the units without a workgroup (32/8 heads; by splits):
//   17 x 3000    1: 58.1/36.7   2: 63.6/39.0   3: 52.8/32.6      17 x 16384   1: 275/150   2: 292/160   3: 234/130
//   22 x 3000    1: 64.2/39.6   2: 70.5/41.6   3: 71.6/43.7      22 x 16384   1: 302/162   2: 316/172   3: 325/176
//   26 x 3000    1: 69.6/42.2   2: 74.6/43.9                     26 x 32768   1: 674/349   2: 695/374
//   28 x 1000    1: 31.6/22.2   2: 34.8/23.0                     28 x 32768   1: 702/377   2: 722/389
//   gather of 26 x 896 rows 1: 20.7  2: 25.2    of 26 x 1664 1: 34.4  2: 39.1    of 17 x 6656 1: 103.6  2: 113.3  3: 88.2  4: 94.5
int kascade_decode_whole_rounds(int lists, double rows, int num_split, int compute_units, double cap_rows) {
    if (lists <= 0 || num_split <= 0) return num_split > 0 ? num_split : 1;
    const double wgs = (double)lists * num_split;
    return wgs > compute_units && wgs < 0.9 * 2 * compute_units ? whole_rounds(lists, rows, num_split, compute_units, cap_rows) : num_split;
}

int kascade_decode_num_split_equal(int lists, double rows, int compute_units, double wgs_per_cu, double min_rows, double cap_rows) {
    int ns = kascade_decode_num_split((double)lists * rows, rows, compute_units, wgs_per_cu, min_rows, cap_rows);
    if (lists <= 0) return ns;
    // Gathers (only small ones come to more than 12): the merge requests 16 splits' results in one trip to memory and pays
    // another for more, which lists of up to about 384 rows a split don't make good.  Us, batch 1, by splits (the last: 128
    // rows each):
    //   3328 rows   32/8 heads 16: 10.2  26: 11.2    64/8 11.9  13.4    28/4 11.1  11.5    8/2 heads of 64 8.1  8.3
    //   6016 rows   28/4 16: 12.7  47: 13.2          8/2 heads of 64 16: 9.2  47: 10.9     64/8 16: 14.5  32: 15.8
    //   8064 rows   32/8 16: 14.7  32: 14.1          11008, 28/4 32: 14.9  64: 14.1
    // Not where the lists may be shorter than the launch has room for: room for 3328 rows, 512 8.7 against 7.5 with 26, 1664 9.5/8.5.
    if (cap_rows > 0 && rows <= 16 * 384 && min_rows >= 384) ns = (int)fmin(ns, 16);
    // Few lists, streamed: one is the better number also where two fill the chip.  Up to 32 lists at any length (batch 1, 32/8
    // heads, two / one: 40000 tokens 54.6/48.9 -> 52.1/48.7 us, 131072 148.7/100.0 -> 142.3/97.7, 180000 174.4/107.6 -> 172.3/104.5,
    // 524288 415.1/233.7 -> 409.8/230.7; 28/4, 262144 144.0/91.9 -> 140.4/91.7; four sequences of 16000 64.8/41.0 -> 63.6/40.8, of
    // 65536 209.0/123.1 -> 209.6/121.3, of 131072 426.3/248.9 -> 421.6/242.3), up to 64 to 4160 rows a unit: eight of 16000
    // 109.9/63.6 -> 106.8/62.5, of 24000 (6000 rows a unit) 155.6/89.5 -> 156.0/87.4, of 32768 200.4/114.3 -> 205.6/114.0.
    // Not where they may be shorter than the launch has room for: room for 131072, 32768 tokens 100.3/72.9 against 80.7/59.7
    // with two.
    const double wgs = (double)lists * ns;
    const bool few = cap_rows <= 0 && (lists <= 32 || (lists <= 64 && lists * rows <= 4160. * compute_units));
    if (few && wgs > compute_units && wgs <= 2 * compute_units) return whole_rounds(lists, rows, ns, compute_units, 0);
    return kascade_decode_whole_rounds(lists, rows, ns, compute_units, cap_rows);
}

// A lone split writes its result itself; merging several costs a trip through device-coherent memory, a
// counter and the way back, the more the more query heads and workgroups there are.  Us per launch in a
// captured graph, one split / as many as kascade_decode_num_split gives, 8 KV heads:
//   rows   batch    1 head      2           4           5           7           8           16 heads per KV head
//   256    1        5.5/6.7     5.5/6.7     5.6/6.9     6.0/7.8     6.1/8.1     6.1/8.1     7.3/11.2
//   384    1        6.8/6.6     6.9/6.8     7.0/7.1     7.4/7.9     7.5/8.1     7.6/8.3     8.6/11.4
//   384    4        7.0/7.1     7.1/7.2     7.3/7.4     7.6/8.2     7.7/8.5     7.8/8.6     8.7/11.8
//   384    8        7.5/7.5     7.5/7.5     7.7/7.7     7.9/8.7     8.1/9.0     8.1/9.0     9.1/12.2
//   512    1        7.9/6.9     8.1/6.7     8.2/6.9     8.5/7.9     8.6/8.2     8.8/8.4     9.8/11.5
//   512    2        8.0/7.1     8.2/7.2     8.3/7.2     8.6/8.4     8.8/8.6     8.8/8.7     9.8/11.8
//   512    8        9.1/8.0     9.2/8.0     9.3/8.2     9.6/9.2     9.7/9.5     9.7/9.6     10.7/12.8
// (At 512 rows one split is up to 5 % behind for 5 to 8 heads; the lists' sums would be split otherwise for that.)
int kascade_gather_lone_rows(int group_size, int lists) {
    if (group_size <= 2) return lists >= 64 ? 384 : 256;
    return group_size >= 8 || (group_size >= 5 && lists >= 16) ? 512 : 384;
}

// One workgroup pools a row's tokens for all query heads of its KV head, four heads at a time, where a
// launch of its own spreads them over the chip: the saved launch stops paying as tokens and heads grow.  Us of an anchor
// pass without output in a captured graph, where a launch costs the host nothing, one launch / two, 8 KV heads, batch 1:
//   tokens   1 head    2          4          5          8          12         16 heads per KV head
//   8192     14.4/15.6 14.6/15.8  15.4/16.6  17.7/18.4  18.3/19.4  20.6/21.7  23.4/26.1
//   10240    18.2/18.6 18.5/19.2  19.0/19.9  22.3/21.5  22.7/23.1  26.1/25.9  29.9/27.9
//   14336    20.3/20.3 20.7/20.7  21.2/21.5  25.8/22.9  26.1/24.9  30.3/27.3  34.8/30.3
//   18432    24.5/24.0 24.7/24.6  25.2/25.2  28.9/26.4  31.0/29.4  35.1/32.0  39.9/34.7
//   20480    26.8/24.9 26.9/25.7  27.4/26.3  32.6/28.0  33.6/30.1  38.4/32.5  44.3/36.1
//   24576    26.9/25.6 27.1/25.9  27.8/26.9  32.9/28.7  33.9/30.8  39.2/33.7  45.0/36.9
//   32768    31.4/29.0 31.7/29.2  32.6/30.2  38.6/31.8  39.7/34.2  46.9/37.2  54.2/40.8
// With many rows the selections fill the chip by themselves: batch 8, 24576 tokens 86.3/87.8 with 2 heads, 98.7/94.9 with 8,
// 122.6/116.3 with 16; 32768 111.3/112.7, 136.0/129.0, 168.6/159.1.
// The limits lie above the crossover of captured passes, for more than four heads per KV head by up to 10000 tokens: an
// eager pass also pays the second launch's way through the host, and one over lists of lengths what makes the rows' budgets
// for it.  With 8192 for those groups, passes over new buffers / among others: serving steps of 8 x 17000 tokens at 64/8 heads
// 417 -> 450 us / 329 -> 329, of 4 x 12000 at 28/4 228 -> 265 / 144.5 -> 144.2; transformers cache, 17000 tokens at 64/8
// heads 340 -> 344 / 136.3 -> 130.2.
int kascade_pool_select_row(int group_size, int rows) {
    return group_size == 3 || group_size == 4 || rows >= 64 ? 24576 : 18432;
}

int kascade_decode_anchor_topk_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K,
                                    const kascade_half* V, const int32_t* cache_seqlens, float* glse,
                                    float* Output_partial, float* row_sums, float* scores, kascade_half* Output,
                                    kascade_half* aggregated_scores, int32_t* out_idx, int32_t* out_rows, int batch,
                                    int kv_stride_tokens, int scores_stride, int num_split, int with_output,
                                    int row_len, int k, int fill_value, float topk_percent, const int32_t* valid_len,
                                    const int32_t* n_sel, void* workspace, const int32_t* block_table, int max_pages,
                                    int page_size, const kascade_strides* kv_strides, const kascade_half* k_new,
                                    const kascade_half* v_new, int32_t* sync_counters, void* stream) {
    Shape sh = kRefShape;
    if (shape && get_shape(shape, &sh)) return -1;
    REQUIRE(out_idx, "decode_anchor_topk: null pointer argument");
    REQUIRE(k > 0 && row_len > 0 && row_len <= scores_stride, "decode_anchor_topk: k > 0 and 0 < row_len <= scores_stride required");
    REQUIRE(!(topk_percent > 0.f) || cache_seqlens, "decode_anchor_topk: topk_percent needs cache_seqlens");
    REQUIRE((long long)batch * sh.G < (1LL << 31), "decode_anchor_topk: too many rows");
    const bool fits = row_len <= KASCADE_POOL_SELECT_ROW;
    REQUIRE(fits || aggregated_scores, "decode_anchor_topk: rows of more than %d tokens need aggregated_scores", KASCADE_POOL_SELECT_ROW);
    const bool counted = !(topk_percent > 0.f) || (valid_len && n_sel);   // what a selection of its own needs is there
    REQUIRE(fits || counted,
            "decode_anchor_topk: rows of more than %d tokens need valid_len and n_sel", KASCADE_POOL_SELECT_ROW);
    TopkRows tr{};
    if (out_rows) {
        REQUIRE(block_table, "decode_anchor_topk: out_rows needs a block table");
        int shift;
        if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
        REQUIRE((long long)max_pages * page_size >= row_len, "decode_anchor_topk: block table shorter than the rows it is to translate");
        tr.out_rows = out_rows; tr.block_table = block_table; tr.max_pages = max_pages;
        tr.page_shift = shift; tr.rows_per_seq = sh.G;
    }
    AnchorSelect sel{};
    sel.one_launch = fits && (row_len <= kascade_pool_select_row(sh.gs, batch * sh.G) || !aggregated_scores || !counted);
    sel.out_idx = out_idx; sel.rows = &tr; sel.row_len = row_len; sel.k = k; sel.fill = fill_value;
    sel.topk_percent = topk_percent; sel.valid_len = valid_len; sel.n_sel = n_sel; sel.workspace = workspace;
    return decode_recompute_paged_impl(sh, Q, K, V, cache_seqlens, glse, Output_partial, row_sums, scores, Output,
                                       aggregated_scores, batch, kv_stride_tokens, scores_stride, num_split, with_output,
                                       block_table, max_pages, page_size, kv_strides, k_new, v_new, sync_counters, &sel,
                                       stream);
}

int64_t kascade_topk_workspace_bytes(int rows, int64_t row_len) {
    return topk_split_workspace_bytes(rows, row_len);
}

int kascade_topk_call(const kascade_half* scores, int32_t* out_idx, int rows, int64_t row_stride,
                      int uniform_len, const int32_t* valid_len, const int32_t* n_sel, int period,
                      int k, int fill_value, void* workspace, void* stream) {
    return kascade_topk_rows_call(scores, out_idx, rows, row_stride, uniform_len, valid_len, n_sel,
                                  period, k, fill_value, workspace, nullptr, nullptr, 0, 1, 1, stream);
}

int kascade_topk_rows_call(const kascade_half* scores, int32_t* out_idx, int rows, int64_t row_stride,
                           int uniform_len, const int32_t* valid_len, const int32_t* n_sel, int period,
                           int k, int fill_value, void* workspace, int32_t* out_rows,
                           const int32_t* block_table, int max_pages, int page_size,
                           int rows_per_sequence, void* stream) {
    REQUIRE(scores && out_idx, "topk: null pointer argument");
    TopkRows tr{};
    if (out_rows) {
        REQUIRE(block_table && rows_per_sequence > 0, "topk: out_rows needs a block table and rows_per_sequence > 0");
        int shift;
        if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
        REQUIRE((long long)max_pages * page_size >= uniform_len,
                "topk: block table shorter than the rows it is to translate");
        tr.out_rows = out_rows; tr.block_table = block_table; tr.max_pages = max_pages;
        tr.page_shift = shift; tr.rows_per_seq = rows_per_sequence;
    }
    REQUIRE(rows >= 0 && k > 0 && row_stride > 0, "topk: rows >= 0, k > 0, row_stride > 0 required");
    REQUIRE(uniform_len >= 0 && uniform_len <= row_stride,
            "topk: uniform_len must be within [0, row_stride]");
    REQUIRE(!(valid_len || n_sel) || period > 0, "topk: period must be > 0 with per-row arrays");
    if (period <= 0) period = 1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return select_rows(H(scores), out_idx, rows, row_stride, uniform_len, valid_len, n_sel, period, k, fill_value, workspace,
                       tr, s);
}

namespace {
inline long long sorted_list_bytes(int rows, int k) {
    return (topk_sort_workspace_bytes(rows, k) + 255) / 256 * 256;
}
}  // namespace

int64_t kascade_topk_sorted_workspace_bytes(int rows, int64_t row_len, int k) {
    if (rows < 0 || k < 0) return 0;
    return sorted_list_bytes(rows, k) + topk_split_workspace_bytes(rows, row_len);
}

int kascade_topk_sorted_call(const kascade_half* scores, int32_t* out_idx, int rows, int64_t row_stride,
                             int uniform_len, const int32_t* valid_len, int period, int k,
                             void* workspace, void* stream) {
    REQUIRE(k > 0 && k <= uniform_len, "topk_sorted: 0 < k <= uniform_len required (as torch.topk)");
    REQUIRE(rows >= 0, "topk_sorted: rows >= 0 required");
    REQUIRE(workspace || kascade_topk_sorted_workspace_bytes(rows, uniform_len, k) == 0,
            "topk_sorted: workspace of kascade_topk_sorted_workspace_bytes() bytes required");
    char* ws = static_cast<char*>(workspace);
    void* split_ws = topk_split_workspace_bytes(rows, uniform_len) > 0 ? ws + sorted_list_bytes(rows, k) : nullptr;
    // the k largest of every row in position order (all valid positions, then the first positions
    // past the row's end, when a row holds fewer than k), then the reordering by score
    if (kascade_topk_call(scores, out_idx, rows, row_stride, uniform_len, valid_len, nullptr, period, k, 0,
                          split_ws, stream))
        return -1;
    if (period <= 0) period = 1;
    return check_hip(launch_topk_sort_rows(H(scores), out_idx, ws, rows, row_stride, uniform_len, valid_len,
                                           period, k, static_cast<hipStream_t>(stream)), "topk_sorted");
}

}  // extern "C"
namespace {
// 64 queries per wavefront in the K-only log-sum pass, or 32?  Units (workgroups) of 64 read every K tile for
// twice the queries, 15 % less per query, but there are half as many and each is twice as long, so it is a
// question of how the units fill the 512 places of the chip (two on each of 256 compute units), and of how
// far their lengths spread: from q_start to q_start + q_len keys.  Us, 32 / 64 queries, 32/8 heads:
//   units of 64   queries, position         32 / 64        why
//   256           2048 at 8192              186 / 209      one workgroup per compute unit
//   448, 512      3584 at 7168, 4096 at 0   347 / 291, 88 / 98: a residency nearly full of units about equally long
//                                           wins; lengths that spread leave its places idle
//   520, 576      4160 at 8320, 4608 at 1152  424 / 464, 169 / 158: equal lengths leave a second residency nearly
//                                           empty, lengths that spread overlap
//   520, 640      4160, 5120 at 0           93.7 / 102.8, 128.8 / 135.9 (whole prompts)
//   768, 1024     6144, 8192 at 0           192 / 174, 315 / 281; at 4 times their length 1550 / 1465, 2725 / 2345
//   704           11 x 512 at 0             28.8 / 34.3    short units: the set-up counts
//   1024          16 x 512 at 0, at 512     37.3 / 40.8, 74.9 / 70.9
// Sequences at different positions count as if all stood at the last one (the host knows no other).
bool wide_log_sum_units(const Shape& sh, int batch, int q_start, int q_len) {
    if (sh.D != 128) return false;
    const long long units = (long long)((q_len + 63) / 64) * sh.G * ((sh.gs + 3) / 4) * batch;
    const bool deep = (long long)q_start + q_len >= 2048;
    if (units <= 512) return units >= 448 && q_start >= q_len;
    if (units <= 640) return deep && q_start > 0 && q_start <= q_len;
    return deep || (q_start >= q_len && units >= 800);
}

int prefill_dense_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K, const kascade_half* V,
                               float* log_sum, kascade_half* Output, int batch, int seq_len,
                               kascade_strides q_strides, kascade_strides kv_strides,
                               int with_output, void* stream) {
    REQUIRE(Q && K, "prefill_dense: null pointer argument");
    REQUIRE(!with_output || (V && Output), "prefill_dense: with_output needs V and Output");
    REQUIRE(with_output || log_sum, "prefill_dense: nothing to compute (no Output, no log_sum)");
    REQUIRE(batch > 0 && seq_len > 0 && batch <= 65535, "prefill_dense: bad batch/seq_len");
    REQUIRE(aligned16(Q) && aligned16(K) && (!with_output || (aligned16(V) && aligned16(Output))),
            "prefill_dense: tensors must be 16-byte aligned");
    if (check_strides(q_strides, "Q") || check_strides(kv_strides, "K/V")) return -1;
    PrefillParams p{};
    p.G = sh.G; p.head_dim = sh.D; p.elem = sh.elem; p.gs = sh.gs;
    p.Q = H(Q); p.K = H(K); p.V = with_output ? H(V) : H(K); p.log_sum = log_sum; p.O = H(Output);
    p.q_sb = q_strides.b; p.q_sl = q_strides.l; p.q_sh = q_strides.h;
    p.k_sb = kv_strides.b; p.k_sl = kv_strides.l; p.k_sh = kv_strides.h;
    p.B = batch; p.L = seq_len; p.Lq = seq_len; p.T = (seq_len + kTile - 1) / kTile;
    const int nqb = (!with_output && wide_log_sum_units(sh, batch, 0, seq_len)) ? 2 : 1;
    return check_hip(launch_prefill_attn(p, false, with_output != 0, nqb, static_cast<hipStream_t>(stream)), "prefill_dense");
}
}  // namespace
extern "C" {

int kascade_prefill_dense_call(const kascade_half* Q, const kascade_half* K, const kascade_half* V,
                               float* log_sum, kascade_half* Output, int batch, int seq_len,
                               kascade_strides q_strides, kascade_strides kv_strides,
                               int with_output, void* stream) {
    return prefill_dense_impl(kRefShape, Q, K, V, log_sum, Output, batch, seq_len, q_strides, kv_strides, with_output, stream);
}

int kascade_prefill_dense_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K, const kascade_half* V,
                               float* log_sum, kascade_half* Output, int batch, int seq_len,
                               kascade_strides q_strides, kascade_strides kv_strides,
                               int with_output, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return prefill_dense_impl(sh, Q, K, V, log_sum, Output, batch, seq_len, q_strides, kv_strides, with_output, stream);
}

}  // extern "C"
namespace {
int prefill_aggregate_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K,
                                   const float* log_sum, kascade_half* aggregate_scores, int batch,
                                   int seq_len, kascade_strides q_strides,
                                   kascade_strides kv_strides, int fill_invalid, void* stream) {
    REQUIRE(Q && K && log_sum && aggregate_scores, "prefill_aggregate: null pointer argument");
    REQUIRE(batch > 0 && seq_len > 0 && batch <= 65535, "prefill_aggregate: bad batch/seq_len");
    REQUIRE(aligned16(Q) && aligned16(K), "prefill_aggregate: Q/K must be 16-byte aligned");
    if (check_strides(q_strides, "Q") || check_strides(kv_strides, "K")) return -1;
    PrefillParams p{};
    p.G = sh.G; p.head_dim = sh.D; p.elem = sh.elem; p.gs = sh.gs;
    p.Q = H(Q); p.K = H(K); p.V = H(K); p.log_sum_in = log_sum; p.agg = H(aggregate_scores);
    p.q_sb = q_strides.b; p.q_sl = q_strides.l; p.q_sh = q_strides.h;
    p.k_sb = kv_strides.b; p.k_sl = kv_strides.l; p.k_sh = kv_strides.h;
    p.B = batch; p.L = seq_len; p.Lq = seq_len; p.T = (seq_len + kTile - 1) / kTile; p.fill_invalid = fill_invalid;
    return check_hip(launch_prefill_aggregate(p, nullptr, static_cast<hipStream_t>(stream)),
                     "prefill_aggregate");
}
}  // namespace
extern "C" {

int kascade_prefill_aggregate_call(const kascade_half* Q, const kascade_half* K,
                                   const float* log_sum, kascade_half* aggregate_scores, int batch,
                                   int seq_len, kascade_strides q_strides,
                                   kascade_strides kv_strides, int fill_invalid, void* stream) {
    return prefill_aggregate_impl(kRefShape, Q, K, log_sum, aggregate_scores, batch, seq_len, q_strides, kv_strides, fill_invalid, stream);
}

int kascade_prefill_aggregate_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K,
                                   const float* log_sum, kascade_half* aggregate_scores, int batch,
                                   int seq_len, kascade_strides q_strides,
                                   kascade_strides kv_strides, int fill_invalid, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return prefill_aggregate_impl(sh, Q, K, log_sum, aggregate_scores, batch, seq_len, q_strides, kv_strides, fill_invalid, stream);
}

}  // extern "C"
namespace {
int range_params(PrefillParams& p, const Shape& sh, const kascade_half* Q, const kascade_half* K, const float* log_sum,
                 kascade_half* aggregate_scores, int batch, int q_start, int q_len, kascade_strides q_strides,
                 kascade_strides kv_strides, int fill_invalid) {
    REQUIRE(Q && K && log_sum && aggregate_scores, "prefill_aggregate_range: null pointer argument");
    REQUIRE(batch > 0 && q_len > 0 && batch <= 65535, "prefill_aggregate_range: bad batch/q_len");
    REQUIRE(q_start >= 0 && q_start % kTile == 0, "prefill_aggregate_range: q_start must be a multiple of 32");
    REQUIRE((long long)q_start + q_len < (1LL << 31), "prefill_aggregate_range: q_start + q_len out of range");
    REQUIRE(aligned16(Q) && aligned16(K), "prefill_aggregate_range: Q/K must be 16-byte aligned");
    if (check_strides(q_strides, "Q") || check_strides(kv_strides, "K")) return -1;
    p.G = sh.G; p.head_dim = sh.D; p.elem = sh.elem; p.gs = sh.gs;
    p.Q = H(Q); p.K = H(K); p.V = H(K); p.log_sum_in = log_sum; p.agg = H(aggregate_scores);
    p.q_sb = q_strides.b; p.q_sl = q_strides.l; p.q_sh = q_strides.h;
    p.k_sb = kv_strides.b; p.k_sl = kv_strides.l; p.k_sh = kv_strides.h;
    p.B = batch; p.L = q_start + q_len; p.Lq = q_len; p.q_start = q_start;
    p.T = (q_len + kTile - 1) / kTile; p.fill_invalid = fill_invalid;
    return 0;
}

int prefill_aggregate_range_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K,
                                         const float* log_sum, kascade_half* aggregate_scores,
                                         int batch, int q_start, int q_len,
                                         kascade_strides q_strides, kascade_strides kv_strides,
                                         int fill_invalid, void* stream) {
    PrefillParams p{};
    if (range_params(p, sh, Q, K, log_sum, aggregate_scores, batch, q_start, q_len, q_strides, kv_strides, fill_invalid)) return -1;
    return check_hip(launch_prefill_aggregate(p, nullptr, static_cast<hipStream_t>(stream)),
                     "prefill_aggregate_range");
}
}  // namespace
extern "C" {

int kascade_prefill_aggregate_range_call(const kascade_half* Q, const kascade_half* K,
                                         const float* log_sum, kascade_half* aggregate_scores,
                                         int batch, int q_start, int q_len,
                                         kascade_strides q_strides, kascade_strides kv_strides,
                                         int fill_invalid, void* stream) {
    return prefill_aggregate_range_impl(kRefShape, Q, K, log_sum, aggregate_scores, batch, q_start, q_len, q_strides, kv_strides, fill_invalid, stream);
}

int kascade_prefill_aggregate_range_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K,
                                         const float* log_sum, kascade_half* aggregate_scores,
                                         int batch, int q_start, int q_len,
                                         kascade_strides q_strides, kascade_strides kv_strides,
                                         int fill_invalid, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return prefill_aggregate_range_impl(sh, Q, K, log_sum, aggregate_scores, batch, q_start, q_len, q_strides, kv_strides, fill_invalid, stream);
}

}  // extern "C"
namespace {
int prefill_reuse_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K, const kascade_half* V,
                               const int32_t* topk_indices, const int32_t* head_mapping,
                               float topk_percent, kascade_half* Output, int batch, int seq_len,
                               int max_topk_num, int rolling, kascade_strides q_strides,
                               kascade_strides kv_strides, float* log_sum, void* stream) {
    REQUIRE(Q && K && V && topk_indices && head_mapping && Output,
            "prefill_reuse: null pointer argument");
    REQUIRE(batch > 0 && seq_len > 0 && batch <= 65535, "prefill_reuse: bad batch/seq_len");
    REQUIRE(max_topk_num > 0, "prefill_reuse: max_topk_num must be > 0");
    REQUIRE(!rolling || topk_percent > 0.f, "prefill_reuse: rolling needs topk_percent > 0");
    REQUIRE(aligned16(Q) && aligned16(K) && aligned16(V) && aligned16(Output),
            "prefill_reuse: tensors must be 16-byte aligned");
    if (check_strides(q_strides, "Q") || check_strides(kv_strides, "K/V")) return -1;
    PrefillParams p{};
    p.G = sh.G; p.head_dim = sh.D; p.elem = sh.elem; p.gs = sh.gs;
    p.Q = H(Q); p.K = H(K); p.V = H(V); p.idx = topk_indices; p.head_map = head_mapping;
    p.O = H(Output); p.log_sum = log_sum;
    p.q_sb = q_strides.b; p.q_sl = q_strides.l; p.q_sh = q_strides.h;
    p.k_sb = kv_strides.b; p.k_sl = kv_strides.l; p.k_sh = kv_strides.h;
    p.B = batch; p.L = seq_len; p.Lq = seq_len; p.T = (seq_len + kTile - 1) / kTile;
    p.max_topk = max_topk_num; p.rolling = rolling; p.topk_percent = topk_percent;
    return check_hip(launch_prefill_attn(p, true, true, 1, static_cast<hipStream_t>(stream)),
                     "prefill_reuse");
}
}  // namespace
extern "C" {

int kascade_prefill_reuse_call(const kascade_half* Q, const kascade_half* K, const kascade_half* V,
                               const int32_t* topk_indices, const int32_t* head_mapping,
                               float topk_percent, kascade_half* Output, int batch, int seq_len,
                               int max_topk_num, int rolling, kascade_strides q_strides,
                               kascade_strides kv_strides, float* log_sum, void* stream) {
    return prefill_reuse_impl(kRefShape, Q, K, V, topk_indices, head_mapping, topk_percent, Output, batch, seq_len, max_topk_num, rolling, q_strides, kv_strides, log_sum, stream);
}

int kascade_prefill_reuse_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K, const kascade_half* V,
                               const int32_t* topk_indices, const int32_t* head_mapping,
                               float topk_percent, kascade_half* Output, int batch, int seq_len,
                               int max_topk_num, int rolling, kascade_strides q_strides,
                               kascade_strides kv_strides, float* log_sum, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return prefill_reuse_impl(sh, Q, K, V, topk_indices, head_mapping, topk_percent, Output, batch, seq_len, max_topk_num, rolling, q_strides, kv_strides, log_sum, stream);
}

}  // extern "C"
namespace {
int paged_kv_append_impl(const Shape& sh, kascade_half* K_pages, kascade_half* V_pages,
                                 const kascade_half* k_new, const kascade_half* v_new,
                                 const int32_t* start_pos, const int32_t* block_table, int batch,
                                 int n_new, int max_pages, int page_size,
                                 kascade_strides new_strides, const int32_t* n_new_rows, void* stream) {
    REQUIRE(K_pages && V_pages && k_new && v_new && start_pos && block_table,
            "paged_kv_append: null pointer argument");
    REQUIRE(batch > 0 && n_new >= 0, "paged_kv_append: bad batch/n_new");
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    REQUIRE(new_strides.b % 8 == 0 && new_strides.l % 8 == 0 && new_strides.h % 8 == 0,
            "paged_kv_append: strides must be multiples of 8 elements");
    REQUIRE(aligned16(K_pages) && aligned16(V_pages) && aligned16(k_new) && aligned16(v_new),
            "paged_kv_append: tensors must be 16-byte aligned");
    return check_hip(launch_paged_kv_append(H(K_pages), H(V_pages), H(k_new), H(v_new), start_pos,
                                            block_table, batch, n_new, n_new_rows, max_pages, shift,
                                            new_strides.b, new_strides.l, new_strides.h, sh.G, sh.D,
                                            static_cast<hipStream_t>(stream)),
                     "paged_kv_append");
}
}  // namespace
extern "C" {

int kascade_paged_kv_append_call(kascade_half* K_pages, kascade_half* V_pages,
                                 const kascade_half* k_new, const kascade_half* v_new,
                                 const int32_t* start_pos, const int32_t* block_table, int batch,
                                 int n_new, int max_pages, int page_size,
                                 kascade_strides new_strides, const int32_t* n_new_rows, void* stream) {
    return paged_kv_append_impl(kRefShape, K_pages, V_pages, k_new, v_new, start_pos, block_table, batch, n_new, max_pages, page_size, new_strides, n_new_rows, stream);
}

int kascade_paged_kv_append_shaped_call(const kascade_shape* shape, kascade_half* K_pages, kascade_half* V_pages,
                                 const kascade_half* k_new, const kascade_half* v_new,
                                 const int32_t* start_pos, const int32_t* block_table, int batch,
                                 int n_new, int max_pages, int page_size,
                                 kascade_strides new_strides, const int32_t* n_new_rows, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return paged_kv_append_impl(sh, K_pages, V_pages, k_new, v_new, start_pos, block_table, batch, n_new, max_pages, page_size, new_strides, n_new_rows, stream);
}

}  // extern "C"
namespace {
int rope_append_impl(const Shape& sh, const kascade_half* q_in, const kascade_strides* q_strides,
                                   const kascade_half* k_in, const kascade_half* v_in,
                                   const kascade_strides* kv_strides, const float* cos_sin,
                                   int max_pos, const kascade_half* q_norm_weight,
                                   const kascade_half* k_norm_weight, float norm_eps,
                                   const int32_t* start_pos, int pos_offset, kascade_half* q_out,
                                   kascade_half* K_pages, kascade_half* V_pages,
                                   const int32_t* block_table, int max_pages, int page_size,
                                   int batch, int n_new, void* stream) {
    REQUIRE(q_in && k_in && v_in && cos_sin && start_pos && q_out && K_pages && V_pages && block_table,
            "rope_append: null pointer argument");
    REQUIRE(batch > 0 && n_new >= 0 && max_pos > 0, "rope_append: bad batch/n_new/max_pos");
    REQUIRE((long long)batch * n_new < (1LL << 31), "rope_append: too many tokens for one launch");
    REQUIRE(norm_eps >= 0.f, "rope_append: norm_eps must not be negative");
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    RopeAppendParams p{};
    const kascade_strides qs = q_strides ? *q_strides
        : kascade_strides{(long long)n_new * sh.H() * sh.D, (long long)sh.H() * sh.D, sh.D};
    const kascade_strides ks = kv_strides ? *kv_strides
        : kascade_strides{(long long)n_new * sh.G * sh.D, (long long)sh.G * sh.D, sh.D};
    if (check_strides(qs, "q_in") || check_strides(ks, "k_in/v_in")) return -1;
    REQUIRE(aligned16(q_in) && aligned16(k_in) && aligned16(v_in) && aligned16(q_out) &&
                aligned16(K_pages) && aligned16(V_pages) && aligned16(cos_sin) &&
                aligned16(q_norm_weight) && aligned16(k_norm_weight),
            "rope_append: tensors must be 16-byte aligned");
    p.q_in = E(q_in); p.k_in = E(k_in); p.v_in = E(v_in);
    p.cos_sin = cos_sin; p.q_weight = E(q_norm_weight); p.k_weight = E(k_norm_weight);
    p.start_pos = start_pos; p.q_out = E(q_out); p.Kp = E(K_pages); p.Vp = E(V_pages);
    p.block_table = block_table;
    p.q_sb = qs.b; p.q_sl = qs.l; p.q_sh = qs.h;
    p.kv_sb = ks.b; p.kv_sl = ks.l; p.kv_sh = ks.h;
    p.eps = norm_eps; p.pos_offset = pos_offset; p.batch = batch; p.n_new = n_new;
    p.max_pages = max_pages; p.page_shift = shift; p.max_pos = max_pos;
    p.G = sh.G; p.head_dim = sh.D; p.elem = sh.elem; p.gs = sh.gs;
    return check_hip(launch_rope_append(p, static_cast<hipStream_t>(stream)), "rope_append");
}
}  // namespace
extern "C" {

int kascade_rope_append_paged_call(const kascade_half* q_in, const kascade_strides* q_strides,
                                   const kascade_half* k_in, const kascade_half* v_in,
                                   const kascade_strides* kv_strides, const float* cos_sin,
                                   int max_pos, const kascade_half* q_norm_weight,
                                   const kascade_half* k_norm_weight, float norm_eps,
                                   const int32_t* start_pos, int pos_offset, kascade_half* q_out,
                                   kascade_half* K_pages, kascade_half* V_pages,
                                   const int32_t* block_table, int max_pages, int page_size,
                                   int batch, int n_new, void* stream) {
    return rope_append_impl(kRefShape, q_in, q_strides, k_in, v_in, kv_strides, cos_sin, max_pos, q_norm_weight, k_norm_weight, norm_eps, start_pos, pos_offset, q_out, K_pages, V_pages, block_table, max_pages, page_size, batch, n_new, stream);
}

int kascade_rope_append_paged_shaped_call(const kascade_shape* shape, const kascade_half* q_in, const kascade_strides* q_strides,
                                   const kascade_half* k_in, const kascade_half* v_in,
                                   const kascade_strides* kv_strides, const float* cos_sin,
                                   int max_pos, const kascade_half* q_norm_weight,
                                   const kascade_half* k_norm_weight, float norm_eps,
                                   const int32_t* start_pos, int pos_offset, kascade_half* q_out,
                                   kascade_half* K_pages, kascade_half* V_pages,
                                   const int32_t* block_table, int max_pages, int page_size,
                                   int batch, int n_new, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return rope_append_impl(sh, q_in, q_strides, k_in, v_in, kv_strides, cos_sin, max_pos, q_norm_weight, k_norm_weight, norm_eps, start_pos, pos_offset, q_out, K_pages, V_pages, block_table, max_pages, page_size, batch, n_new, stream);
}

int kascade_decode_budgets_shaped_call(const kascade_shape* shape, int32_t* cache_seqlens, int advance,
                                       float topk_percent, int batch, int32_t* valid_len_rows,
                                       int32_t* n_sel_rows, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    REQUIRE(cache_seqlens, "decode_budgets: null pointer argument");
    REQUIRE(batch > 0 && batch <= 65535, "decode_budgets: bad batch");
    REQUIRE(topk_percent >= 0.f && topk_percent <= 100.f, "decode_budgets: topk_percent out of range");
    return check_hip(launch_decode_budgets(cache_seqlens, advance, topk_percent, batch, sh.G, valid_len_rows,
                                           n_sel_rows, static_cast<hipStream_t>(stream)),
                     "decode_budgets");
}

int kascade_decode_budgets_call(int32_t* cache_seqlens, int advance, float topk_percent, int batch,
                                int32_t* valid_len_rows, int32_t* n_sel_rows, void* stream) {
    const kascade_shape ref{kRefShape.G, kRefShape.D, KASCADE_F16, kRefShape.gs};
    return kascade_decode_budgets_shaped_call(&ref, cache_seqlens, advance, topk_percent, batch,
                                              valid_len_rows, n_sel_rows, stream);
}

// ---- chunked prefill over the paged cache ----

}  // extern "C"
namespace {
int chunk_params(PrefillParams& p, const Shape& sh, const kascade_half* Q, int batch,
                        int q_start, int q_len, kascade_strides q_strides,
                        const int32_t* block_table, int max_pages, int page_size, int num_pages,
                        const int32_t* q_start_rows, const int32_t* q_len_rows) {
    REQUIRE(block_table, "prefill_chunk: block_table is required");
    REQUIRE(batch > 0 && batch <= 65535 && q_len > 0, "prefill_chunk: bad batch/q_len");
    REQUIRE(q_start >= 0 && q_start % kTile == 0, "prefill_chunk: q_start must be a multiple of 32");
    REQUIRE(aligned16(Q), "prefill_chunk: Q must be 16-byte aligned");
    if (check_strides(q_strides, "Q")) return -1;
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    REQUIRE(page_size >= 4, "prefill_chunk: page_size must be at least 4");
    REQUIRE(num_pages > 0 && (long long)num_pages * page_size < (1LL << 31),
            "prefill_chunk: num_pages out of range");
    REQUIRE((long long)max_pages * page_size >= (long long)q_start + q_len,
            "prefill_chunk: block table shorter than q_start + q_len");
    p.G = sh.G; p.head_dim = sh.D; p.elem = sh.elem; p.gs = sh.gs;
    p.Q = E(Q);
    p.q_sb = q_strides.b; p.q_sl = q_strides.l; p.q_sh = q_strides.h;
    p.B = batch; p.L = q_start + q_len; p.Lq = q_len; p.q_start = q_start;
    p.T = (q_len + kTile - 1) / kTile;
    p.block_table = block_table; p.max_pages = max_pages; p.page_shift = shift;
    p.num_pages = num_pages;
    REQUIRE(q_start_rows || !q_len_rows, "prefill_chunk: q_len_rows comes with q_start_rows");
    p.q_start_rows = q_start_rows; p.q_len_rows = q_len_rows;
    return 0;
}

int prefill_chunk_dense_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K_pages,
                                     const kascade_half* V_pages, float* log_sum,
                                     kascade_half* Output, int batch, int q_start, int q_len,
                                     kascade_strides q_strides, const int32_t* block_table,
                                     int max_pages, int page_size, int num_pages, int with_output, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows,
                                     void* stream) {
    REQUIRE(Q && K_pages, "prefill_chunk_dense: null pointer argument");
    REQUIRE(!with_output || (V_pages && Output), "prefill_chunk_dense: with_output needs V and Output");
    REQUIRE(with_output || log_sum, "prefill_chunk_dense: nothing to compute (no Output, no log_sum)");
    REQUIRE(aligned16(K_pages) && (!with_output || (aligned16(V_pages) && aligned16(Output))),
            "prefill_chunk_dense: tensors must be 16-byte aligned");
    PrefillParams p{};
    if (chunk_params(p, sh, Q, batch, q_start, q_len, q_strides, block_table, max_pages,
                     page_size, num_pages, q_start_rows, q_len_rows))
        return -1;
    p.K = E(K_pages); p.V = with_output ? E(V_pages) : E(K_pages);
    p.log_sum = log_sum; p.O = E(Output);
    const int nqb = (!with_output && wide_log_sum_units(sh, batch, q_start, q_len)) ? 2 : 1;
    return check_hip(launch_prefill_attn(p, false, with_output != 0, nqb,
                                         static_cast<hipStream_t>(stream)), "prefill_chunk_dense");
}

int prefill_chunk_aggregate_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K_pages,
                                         const float* log_sum, kascade_half* aggregate_scores,
                                         int batch, int q_start, int q_len,
                                         kascade_strides q_strides, const int32_t* block_table,
                                         int max_pages, int page_size, int num_pages,
                                         int fill_invalid, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows, void* stream) {
    REQUIRE(Q && K_pages && log_sum && aggregate_scores,
            "prefill_chunk_aggregate: null pointer argument");
    REQUIRE(aligned16(K_pages), "prefill_chunk_aggregate: K must be 16-byte aligned");
    PrefillParams p{};
    if (chunk_params(p, sh, Q, batch, q_start, q_len, q_strides, block_table, max_pages,
                     page_size, num_pages, q_start_rows, q_len_rows))
        return -1;
    p.K = E(K_pages); p.V = E(K_pages); p.log_sum_in = log_sum; p.agg = H(aggregate_scores);
    p.fill_invalid = fill_invalid;
    return check_hip(launch_prefill_aggregate(p, nullptr, static_cast<hipStream_t>(stream)),
                     "prefill_chunk_aggregate");
}

int prefill_chunk_reuse_impl(const Shape& sh, const kascade_half* Q, const kascade_half* K_pages,
                                     const kascade_half* V_pages, const int32_t* physical_rows,
                                     const int32_t* head_mapping, float topk_percent,
                                     kascade_half* Output, int batch, int q_start, int q_len,
                                     int max_topk_num, int rolling, kascade_strides q_strides,
                                     const int32_t* block_table, int max_pages, int page_size,
                                     int num_pages, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows, float* log_sum, void* stream) {
    REQUIRE(Q && K_pages && V_pages && physical_rows && head_mapping && Output,
            "prefill_chunk_reuse: null pointer argument");
    REQUIRE(max_topk_num > 0, "prefill_chunk_reuse: max_topk_num must be > 0");
    REQUIRE(!rolling || topk_percent > 0.f, "prefill_chunk_reuse: rolling needs topk_percent > 0");
    REQUIRE(aligned16(K_pages) && aligned16(V_pages) && aligned16(Output),
            "prefill_chunk_reuse: tensors must be 16-byte aligned");
    PrefillParams p{};
    if (chunk_params(p, sh, Q, batch, q_start, q_len, q_strides, block_table, max_pages,
                     page_size, num_pages, q_start_rows, q_len_rows))
        return -1;
    p.K = E(K_pages); p.V = E(V_pages); p.idx = physical_rows; p.head_map = head_mapping;
    p.O = E(Output); p.log_sum = log_sum;
    p.max_topk = max_topk_num; p.rolling = rolling; p.topk_percent = topk_percent;
    return check_hip(launch_prefill_attn(p, true, true, 1, static_cast<hipStream_t>(stream)),
                     "prefill_chunk_reuse");
}
}  // namespace
extern "C" {

int kascade_prefill_pool_selects(int kv_heads, int head_dim, int batch, int q_start, int q_len) {
    if (kv_heads < 1 || batch < 1 || q_start < 0 || q_len < 1 || (long long)q_start + q_len >= (1LL << 31)) return 0;
    PrefillParams p{};
    p.G = kv_heads; p.head_dim = head_dim; p.B = batch; p.q_start = q_start; p.T = (q_len + kTile - 1) / kTile;
    return prefill_pool_selects(p) ? 1 : 0;
}

int kascade_prefill_anchor_topk_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K, const float* log_sum,
                                     kascade_half* scores, int32_t* out_idx, int32_t* out_rows, int batch, int q_start, int q_len,
                                     kascade_strides q_strides, const kascade_strides* kv_strides, const int32_t* block_table,
                                     int max_pages, int page_size, int num_pages, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows, const int32_t* valid_len, const int32_t* n_sel, int period, int k,
                                     int fill_value, void* workspace, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    REQUIRE(Q && K && log_sum && scores && out_idx && valid_len && n_sel, "prefill_anchor_topk: null pointer argument");
    REQUIRE(block_table || kv_strides, "prefill_anchor_topk: K is strided or behind a block table");
    REQUIRE(!out_rows || block_table, "prefill_anchor_topk: out_rows needs a block table");
    REQUIRE(k > 0 && period > 0, "prefill_anchor_topk: k and period must be > 0");
    const hipStream_t s = static_cast<hipStream_t>(stream);
    PrefillParams p{};
    if (block_table) {
        REQUIRE(aligned16(K), "prefill_anchor_topk: K must be 16-byte aligned");
        if (chunk_params(p, sh, Q, batch, q_start, q_len, q_strides, block_table, max_pages, page_size, num_pages, q_start_rows,
                         q_len_rows))
            return -1;
        p.K = E(K); p.V = E(K); p.log_sum_in = log_sum; p.agg = H(scores);
    } else {
        REQUIRE(!q_start_rows && !q_len_rows, "prefill_anchor_topk: rows of their own come with a block table");
        if (range_params(p, sh, Q, K, log_sum, scores, batch, q_start, q_len, q_strides, *kv_strides, 0)) return -1;
    }
    const long long rows = (long long)p.B * p.G * p.T;
    REQUIRE(rows < (1LL << 31), "prefill_anchor_topk: too many rows");
    TopkRows tr{};
    if (out_rows) {
        tr.out_rows = out_rows; tr.block_table = block_table; tr.max_pages = max_pages; tr.page_shift = p.page_shift;
        tr.rows_per_seq = p.G * p.T;
    }
    if (prefill_pool_selects(p)) {
        SelectParams sel{valid_len, n_sel, out_idx, tr, period, k, fill_value};
        return check_hip(launch_prefill_aggregate(p, &sel, s), "prefill_anchor_topk");
    }
    if (check_hip(launch_prefill_aggregate(p, nullptr, s), "prefill_anchor_topk")) return -1;
    return select_rows(p.agg, out_idx, (int)rows, p.L, p.L, valid_len, n_sel, period, k, fill_value, workspace, tr, s);
}

int kascade_prefill_chunk_dense_call(const kascade_half* Q, const kascade_half* K_pages,
                                     const kascade_half* V_pages, float* log_sum,
                                     kascade_half* Output, int batch, int q_start, int q_len,
                                     kascade_strides q_strides, const int32_t* block_table,
                                     int max_pages, int page_size, int num_pages, int with_output, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows,
                                     void* stream) {
    return prefill_chunk_dense_impl(kRefShape, Q, K_pages, V_pages, log_sum, Output, batch, q_start, q_len, q_strides, block_table, max_pages, page_size, num_pages, with_output, q_start_rows, q_len_rows, stream);
}

int kascade_prefill_chunk_dense_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K_pages,
                                     const kascade_half* V_pages, float* log_sum,
                                     kascade_half* Output, int batch, int q_start, int q_len,
                                     kascade_strides q_strides, const int32_t* block_table,
                                     int max_pages, int page_size, int num_pages, int with_output, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows,
                                     void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return prefill_chunk_dense_impl(sh, Q, K_pages, V_pages, log_sum, Output, batch, q_start, q_len, q_strides, block_table, max_pages, page_size, num_pages, with_output, q_start_rows, q_len_rows, stream);
}

int kascade_prefill_chunk_aggregate_call(const kascade_half* Q, const kascade_half* K_pages,
                                         const float* log_sum, kascade_half* aggregate_scores,
                                         int batch, int q_start, int q_len,
                                         kascade_strides q_strides, const int32_t* block_table,
                                         int max_pages, int page_size, int num_pages,
                                         int fill_invalid, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows, void* stream) {
    return prefill_chunk_aggregate_impl(kRefShape, Q, K_pages, log_sum, aggregate_scores, batch, q_start, q_len, q_strides, block_table, max_pages, page_size, num_pages, fill_invalid, q_start_rows, q_len_rows, stream);
}

int kascade_prefill_chunk_aggregate_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K_pages,
                                         const float* log_sum, kascade_half* aggregate_scores,
                                         int batch, int q_start, int q_len,
                                         kascade_strides q_strides, const int32_t* block_table,
                                         int max_pages, int page_size, int num_pages,
                                         int fill_invalid, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return prefill_chunk_aggregate_impl(sh, Q, K_pages, log_sum, aggregate_scores, batch, q_start, q_len, q_strides, block_table, max_pages, page_size, num_pages, fill_invalid, q_start_rows, q_len_rows, stream);
}

int kascade_prefill_chunk_reuse_call(const kascade_half* Q, const kascade_half* K_pages,
                                     const kascade_half* V_pages, const int32_t* physical_rows,
                                     const int32_t* head_mapping, float topk_percent,
                                     kascade_half* Output, int batch, int q_start, int q_len,
                                     int max_topk_num, int rolling, kascade_strides q_strides,
                                     const int32_t* block_table, int max_pages, int page_size,
                                     int num_pages, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows, float* log_sum, void* stream) {
    return prefill_chunk_reuse_impl(kRefShape, Q, K_pages, V_pages, physical_rows, head_mapping, topk_percent, Output, batch, q_start, q_len, max_topk_num, rolling, q_strides, block_table, max_pages, page_size, num_pages, q_start_rows, q_len_rows, log_sum, stream);
}

int kascade_prefill_chunk_reuse_shaped_call(const kascade_shape* shape, const kascade_half* Q, const kascade_half* K_pages,
                                     const kascade_half* V_pages, const int32_t* physical_rows,
                                     const int32_t* head_mapping, float topk_percent,
                                     kascade_half* Output, int batch, int q_start, int q_len,
                                     int max_topk_num, int rolling, kascade_strides q_strides,
                                     const int32_t* block_table, int max_pages, int page_size,
                                     int num_pages, const int32_t* q_start_rows,
                                     const int32_t* q_len_rows, float* log_sum, void* stream) {
    Shape sh;
    if (get_shape(shape, &sh)) return -1;
    return prefill_chunk_reuse_impl(sh, Q, K_pages, V_pages, physical_rows, head_mapping, topk_percent, Output, batch, q_start, q_len, max_topk_num, rolling, q_strides, block_table, max_pages, page_size, num_pages, q_start_rows, q_len_rows, log_sum, stream);
}

int kascade_translate_indices_call(const int32_t* token_idx, int32_t* physical_rows,
                                   const int32_t* block_table, int batch, int64_t per_sequence,
                                   int max_pages, int page_size, int kv_len, void* stream) {
    REQUIRE(token_idx && physical_rows && block_table, "translate_indices: null pointer argument");
    REQUIRE(batch > 0 && batch <= 65535 && per_sequence >= 0 && kv_len > 0,
            "translate_indices: bad batch/per_sequence/kv_len");
    int shift;
    if (check_paging(block_table, max_pages, page_size, &shift)) return -1;
    REQUIRE((long long)max_pages * page_size >= kv_len,
            "translate_indices: block table shorter than kv_len");
    return check_hip(launch_translate_indices(token_idx, physical_rows, block_table, batch,
                                              per_sequence, max_pages, shift, kv_len,
                                              static_cast<hipStream_t>(stream)),
                     "translate_indices");
}

// ---- the reference's argument lists, verbatim ----

int kascade_ref_decode_reuse_call(kascade_half* Q, kascade_half* K, kascade_half* V,
                                  int* topk_indices, int* head_mapping, float* glse,
                                  float* Output_partial, kascade_half* Output, int batch,
                                  int kv_seqlen, int topk, void* stream) {
    return kascade_decode_reuse_call(Q, K, V, topk_indices, head_mapping, glse, Output_partial, Output,
                                     batch, kv_seqlen, topk, kRefNumSplit, nullptr, stream);
}

int kascade_ref_decode_reuse_kvcache_call(kascade_half* Q, kascade_half* K, kascade_half* V,
                                          int* cache_seqlens, int* topk_indices, int* head_mapping,
                                          float topk_percent, float* glse, float* Output_partial,
                                          kascade_half* Output, int batch, int max_cache_seqlen,
                                          int topk, void* stream) {
    return kascade_decode_reuse_paged_call(Q, K, V, cache_seqlens, topk_indices, head_mapping,
                                           topk_percent, glse, Output_partial, Output, batch,
                                           max_cache_seqlen, topk, kRefNumSplit, nullptr, 0, 1, nullptr,
                                           nullptr, nullptr, nullptr, nullptr, stream);
}

int kascade_ref_prefill_aggregate_call(kascade_half* Q, kascade_half* K, float* log_sum,
                                       kascade_half* aggregate_scores, int batch, int seq_len,
                                       void* stream) {
    return kascade_prefill_aggregate_call(Q, K, log_sum, aggregate_scores, batch, seq_len,
                                          contiguous_strides(seq_len, kHeads), contiguous_strides(seq_len, kGroups),
                                          0, stream);
}

int kascade_ref_prefill_reuse_rolling_call(kascade_half* Q, kascade_half* K, kascade_half* V,
                                           int* topk_indices, int* head_mapping,
                                           float topk_percent, kascade_half* Output, int batch,
                                           int seq_len, int max_topk_num, void* stream) {
    return kascade_prefill_reuse_call(Q, K, V, topk_indices, head_mapping, topk_percent, Output, batch,
                                      seq_len, max_topk_num, 1, contiguous_strides(seq_len, kHeads),
                                      contiguous_strides(seq_len, kGroups), nullptr, stream);
}

int kascade_ref_prefill_reuse_call(kascade_half* Q, kascade_half* K, kascade_half* V,
                                   int* topk_indices, int* head_mapping, float topk_percent,
                                   kascade_half* Output, int batch, int seq_len, int topk_num,
                                   void* stream) {
    return kascade_prefill_reuse_call(Q, K, V, topk_indices, head_mapping, topk_percent, Output, batch,
                                      seq_len, topk_num, 0, contiguous_strides(seq_len, kHeads),
                                      contiguous_strides(seq_len, kGroups), nullptr, stream);
}

// ---- diagnostics ----

int kascade_diag_stream_read_call(const void* src, int64_t bytes, void* sink, void* stream) {
    REQUIRE(src && sink, "diag_stream_read: null pointer argument");
    REQUIRE(bytes >= 16 && aligned16(src) && aligned16(sink), "diag_stream_read: need >= 16 bytes, 16-byte aligned");
    const int cus = g_cu_count > 0 ? g_cu_count : 256;
    return check_hip(launch_diag_stream_read(src, bytes, sink, cus * 32, static_cast<hipStream_t>(stream)),
                     "diag_stream_read");
}

int kascade_diag_gather_rows_call(const void* rows_a, const void* rows_b, const int32_t* row_ids,
                                  int64_t n_rows, int64_t row_stride_bytes, void* sink, void* stream) {
    REQUIRE(rows_a && row_ids && sink, "diag_gather_rows: null pointer argument");
    REQUIRE(n_rows > 0 && row_stride_bytes >= 256 && row_stride_bytes % 16 == 0,
            "diag_gather_rows: n_rows > 0 and a row stride of at least 256 bytes, multiple of 16, required");
    REQUIRE(aligned16(rows_a) && (!rows_b || aligned16(rows_b)) && aligned16(sink),
            "diag_gather_rows: arrays must be 16-byte aligned");
    return check_hip(launch_diag_gather_rows(rows_a, rows_b, row_ids, n_rows, 128, row_stride_bytes, sink,
                                             static_cast<hipStream_t>(stream)), "diag_gather_rows");
}

}  // extern "C"
