// C-ABI of the ETHOS expert-layer kernels (declared in include/ethos_hip.h).
// Every entry point validates its arguments, enqueues on the caller's stream, never
// allocates, never throws, and returns 0 on success, a negative ETHOS_E* code for an
// argument error, or a positive hipError_t; ethos_last_error() describes the last
// failure of the calling thread.
#include <stdarg.h>
#include <stdio.h>

#include <atomic>

#include "../../include/ethos_hip.h"
#include "ethos_common.hpp"
#include "ethos_launch.hpp"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int hip_status(int rc, const char* what) {
    if (rc == 0) return 0;
    return fail(rc, "%s: %s", what, hipGetErrorString((hipError_t)rc));
}

constexpr int kMaxDevices = 64;
std::atomic<int> g_num_cus[kMaxDevices];

int num_cus() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
    int n = g_num_cus[dev].load(std::memory_order_relaxed);
    if (n <= 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        g_num_cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }
bool dtype_ok(int dtype) { return dtype == ETHOS_F32 || dtype == ETHOS_BF16; }

// Sort workspace of ethos_sort_segment_noalloc: one array per GPU, in the code object's
// device data, sized for ETHOS_NOALLOC_MAX_PAIRS pairs (a batch that size sorts without
// the expert -> slot table).  Its name is only a host-side
// stand-in; kernels receive the device address that hipGetSymbolAddress returns for the
// current device (g_scratch_ptr), looked up once per device on the first call there.
constexpr size_t kScratchWords = ethos::sort_workspace_words(ETHOS_NOALLOC_MAX_PAIRS, (int64_t)1 << 18);
static __device__ __align__(256) uint32_t scratch[kScratchWords];
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (nullptr and the error in g_err on failure).
void* scratch_ptr(int* rc) {
    int dev = 0;
    *rc = (int)hipGetDevice(&dev);
    if (*rc != 0) {
        fail(*rc, "ethos_sort_segment_noalloc: hipGetDevice: %s", hipGetErrorString((hipError_t)*rc));
        return nullptr;
    }
    if (dev < 0 || dev >= kMaxDevices) {
        *rc = ETHOS_EUNSUPPORTED;
        fail(*rc, "ethos_sort_segment_noalloc: device %d beyond the %d this library tracks", dev, kMaxDevices);
        return nullptr;
    }
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (p) return p;
    *rc = (int)hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (*rc != 0 || !p) {
        if (*rc == 0) *rc = (int)hipErrorInvalidSymbol;
        fail(*rc, "ethos_sort_segment_noalloc: hipGetSymbolAddress(scratch): %s", hipGetErrorString((hipError_t)*rc));
        return nullptr;
    }
    g_scratch_ptr[dev].store(p, std::memory_order_release);
    return p;
}

// Stage events of the calling thread (ethos_stage_events): recorded in order, one per
// stage boundary, until the list is used up.
thread_local hipEvent_t g_events[16];
thread_local int g_n_events = 0, g_next_event = 0;

}  // namespace

namespace ethos {
void stage_mark(hipStream_t stream) {
    if (g_next_event < g_n_events) (void)hipEventRecord(g_events[g_next_event++], stream);
}
}  // namespace ethos

extern "C" {

int ethos_stage_events(void* const* events, int32_t n_events) {
    g_err[0] = 0;
    if (n_events < 0 || n_events > 16 || (n_events > 0 && !events))
        return fail(ETHOS_ESIZE, "ethos_stage_events: 0 to 16 events, got %d", n_events);
    for (int i = 0; i < n_events; ++i) {
        if (!events[i]) return fail(ETHOS_ENULL, "ethos_stage_events: event %d is NULL", i);
        g_events[i] = (hipEvent_t)events[i];
    }
    g_n_events = n_events;
    g_next_event = 0;
    return 0;
}

const char* ethos_last_error(void) { return g_err; }

int ethos_abi_version(void) { return ETHOS_ABI_VERSION; }

size_t ethos_query_proj_workspace_bytes(int64_t n_tok, int32_t d_model, int32_t n_heads, int32_t d_query,
                                        int32_t dtype) {
    if (n_tok <= 0 || d_model <= 0 || n_heads <= 0 || d_query <= 0) return 256;
    const size_t b = ethos::qproj_workspace_bytes(n_tok, n_heads * d_query, d_model, dtype);
    return b < 256 ? 256 : b;
}

static int query_proj_checks(const char* name, const void* x, const void* wq, const void* prepared, const void* bq,
                             const float* bn_alpha, const float* bn_beta, int64_t n_tok, int32_t d_model,
                             int32_t n_heads, int32_t d_query, int32_t dtype, const void* workspace,
                             size_t workspace_bytes, const void* q_out) {
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "%s: unknown dtype %d", name, dtype);
    if (n_tok < 0 || d_model <= 0 || n_heads <= 0 || d_query <= 0)
        return fail(ETHOS_ESIZE, "%s: bad sizes n_tok=%lld d_model=%d n_heads=%d d_query=%d", name,
                    (long long)n_tok, d_model, n_heads, d_query);
    if ((int64_t)n_heads * d_query > INT32_MAX / 2 || n_tok * (int64_t)n_heads * d_query > INT32_MAX)
        return fail(ETHOS_ESIZE, "%s: n_tok * n_heads * d_query exceeds int32", name);
    if (n_tok == 0) return 0;
    if (!x || !wq || !bq || !bn_alpha || !bn_beta || !q_out) return fail(ETHOS_ENULL, "%s: null pointer", name);
    const size_t need = ethos_query_proj_workspace_bytes(n_tok, d_model, n_heads, d_query, dtype);
    if (dtype == ETHOS_BF16) {
        if (!workspace || workspace_bytes < need)
            return fail(ETHOS_EWORKSPACE, "%s: workspace of %zu bytes, %zu needed", name, workspace_bytes, need);
        if (!aligned16(workspace) || !aligned16(x) || !aligned16(wq) || (prepared && !aligned16(prepared)) ||
            (d_model % 8))
            return fail(ETHOS_EALIGN, "%s: x, wq, prepared, workspace 16-byte aligned and d_model %% 8 == 0", name);
    }
    return 0;
}

static int query_proj_impl(const char* name, const void* x, const void* wq, const void* prepared, const void* bq,
                           const float* bn_alpha, const float* bn_beta, int64_t n_tok, int32_t d_model,
                           int32_t n_heads, int32_t d_query, int32_t dtype, void* workspace, size_t workspace_bytes,
                           void* q_out, void* stream) {
    g_err[0] = 0;
    if (const int rc = query_proj_checks(name, x, wq, prepared, bq, bn_alpha, bn_beta, n_tok, d_model, n_heads, d_query, dtype,
                                         workspace, workspace_bytes, q_out))
        return rc;
    if (n_tok == 0) return 0;
    if (ethos::qproj_weights_bytes(n_heads * d_query, d_model, dtype) == 0) prepared = nullptr;
    return hip_status(ethos::launch_qproj(x, wq, prepared, bq, bn_alpha, bn_beta, n_tok, d_model, n_heads * d_query,
                                          dtype, workspace, q_out, num_cus(), (hipStream_t)stream),
                      name);
}

int ethos_query_proj(const void* x, const void* wq, const void* bq, const float* bn_alpha, const float* bn_beta,
                     int64_t n_tok, int32_t d_model, int32_t n_heads, int32_t d_query, int32_t dtype, void* workspace,
                     size_t workspace_bytes, void* q_out, void* stream) {
    return query_proj_impl("ethos_query_proj", x, wq, nullptr, bq, bn_alpha, bn_beta, n_tok, d_model, n_heads,
                           d_query, dtype, workspace, workspace_bytes, q_out, stream);
}

size_t ethos_query_proj_weights_bytes(int32_t d_model, int32_t n_heads, int32_t d_query, int32_t dtype) {
    if (d_model <= 0 || n_heads <= 0 || d_query <= 0 || !dtype_ok(dtype)) return 0;
    return ethos::qproj_weights_bytes(n_heads * d_query, d_model, dtype);
}

int ethos_query_proj_prepare(const void* wq, int32_t d_model, int32_t n_heads, int32_t d_query, int32_t dtype,
                             void* prepared, size_t prepared_bytes, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_query_proj_prepare: unknown dtype %d", dtype);
    if (d_model <= 0 || n_heads <= 0 || d_query <= 0 || (int64_t)n_heads * d_query > INT32_MAX / 2)
        return fail(ETHOS_ESIZE, "ethos_query_proj_prepare: bad sizes d_model=%d n_heads=%d d_query=%d", d_model,
                    n_heads, d_query);
    const size_t need = ethos_query_proj_weights_bytes(d_model, n_heads, d_query, dtype);
    if (need == 0) return 0;
    if (!wq || !prepared) return fail(ETHOS_ENULL, "ethos_query_proj_prepare: null pointer");
    if (prepared_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_query_proj_prepare: %zu bytes, %zu needed", prepared_bytes, need);
    if (!aligned16(wq) || !aligned16(prepared) || (d_model % 8))
        return fail(ETHOS_EALIGN, "ethos_query_proj_prepare: wq, prepared 16-byte aligned and d_model %% 8 == 0");
    return hip_status(ethos::launch_qproj_prepare(wq, n_heads * d_query, d_model, dtype, prepared,
                                                  (hipStream_t)stream),
                      "ethos_query_proj_prepare");
}

static int query_prepared_checks(const char* name, const void* prepared, size_t prepared_bytes, int64_t n_tok, int32_t d_model,
                                 int32_t n_heads, int32_t d_query, int32_t dtype) {
    const size_t need = ethos_query_proj_weights_bytes(d_model, n_heads, d_query, dtype);
    if (need > 0 && n_tok > 0) {
        if (!prepared) return fail(ETHOS_ENULL, "%s: null prepared weights", name);
        if (prepared_bytes < need)
            return fail(ETHOS_EWORKSPACE, "%s: prepared weights of %zu bytes, %zu needed", name, prepared_bytes, need);
    }
    return 0;
}

int ethos_query_proj_prepared(const void* x, const void* wq, const void* prepared, size_t prepared_bytes,
                              const void* bq, const float* bn_alpha, const float* bn_beta, int64_t n_tok,
                              int32_t d_model, int32_t n_heads, int32_t d_query, int32_t dtype, void* workspace,
                              size_t workspace_bytes, void* q_out, void* stream) {
    g_err[0] = 0;
    if (const int rc = query_prepared_checks("ethos_query_proj_prepared", prepared, prepared_bytes, n_tok, d_model, n_heads,
                                             d_query, dtype))
        return rc;
    return query_proj_impl("ethos_query_proj_prepared", x, wq, prepared, bq, bn_alpha, bn_beta, n_tok, d_model,
                           n_heads, d_query, dtype, workspace, workspace_bytes, q_out, stream);
}

static int route_checks(const char* name, int64_t n_rows, int32_t d_query, int32_t n_sub_keys, int32_t top_k,
                        int32_t k_cand, int32_t dtype) {
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "%s: unknown dtype %d", name, dtype);
    if (n_rows < 0 || d_query <= 0 || (d_query & 1) || n_sub_keys <= 0 || top_k <= 0 || k_cand <= 0)
        return fail(ETHOS_ESIZE, "%s: bad sizes rows=%lld d_query=%d K=%d top_k=%d k_cand=%d", name,
                    (long long)n_rows, d_query, n_sub_keys, top_k, k_cand);
    if (k_cand > n_sub_keys) return fail(ETHOS_ESIZE, "%s: k_cand=%d exceeds the %d sub-keys", name, k_cand, n_sub_keys);
    if (top_k > k_cand * k_cand) return fail(ETHOS_ESIZE, "%s: top_k=%d exceeds k_cand^2=%d", name, top_k, k_cand * k_cand);
    if (k_cand > 32 || top_k > 32)
        return fail(ETHOS_EUNSUPPORTED, "%s: k_cand=%d / top_k=%d above 32 are not supported", name, k_cand, top_k);
    if ((int64_t)n_sub_keys * n_sub_keys > INT32_MAX)
        return fail(ETHOS_EUNSUPPORTED, "%s: %d sub-keys give expert ids beyond int32", name, n_sub_keys);
    if (!ethos::route_supported(n_sub_keys, d_query / 2, dtype))
        return fail(ETHOS_EUNSUPPORTED,
                    "%s: needs n_sub_keys <= 512, d_query/2 <= 256 and d_query/2 %% %d == 0 (got %d, %d)", name,
                    dtype == ETHOS_BF16 ? 16 : 4, n_sub_keys, d_query);
    return 0;
}

static int route_pointer_checks(const char* name, const void* q, const void* sub_keys_1, const void* sub_keys_2,
                                const void* out_scores, const void* out_ids) {
    if (!q || !sub_keys_1 || !sub_keys_2 || !out_scores || !out_ids) return fail(ETHOS_ENULL, "%s: null pointer", name);
    if (!aligned16(q) || !aligned16(sub_keys_1) || !aligned16(sub_keys_2))
        return fail(ETHOS_EALIGN, "%s: q and sub-key tables must be 16-byte aligned", name);
    return 0;
}

static int route_prepared_checks(const char* name, const void* prepared, size_t prepared_bytes, int32_t d_query,
                                 int32_t n_sub_keys, int32_t dtype) {
    if (!prepared) return fail(ETHOS_ENULL, "%s: null pointer", name);
    const size_t need = ethos::route_keys_bytes(n_sub_keys, d_query / 2, dtype);
    if (prepared_bytes < need) return fail(ETHOS_ESIZE, "%s: prepared holds %zu bytes, needs %zu", name, prepared_bytes, need);
    if (!aligned16(prepared)) return fail(ETHOS_EALIGN, "%s: prepared must be 16-byte aligned", name);
    return 0;
}

int ethos_route_topk(const void* q, const void* sub_keys_1, const void* sub_keys_2, const float* key_norms,
                     int64_t n_rows, int32_t d_query, int32_t n_sub_keys, int32_t top_k, int32_t k_cand, int32_t dtype,
                     void* out_scores, int32_t* out_ids, void* stream) {
    g_err[0] = 0;
    if (const int rc = route_checks("ethos_route_topk", n_rows, d_query, n_sub_keys, top_k, k_cand, dtype)) return rc;
    if (n_rows == 0) return 0;
    if (const int rc = route_pointer_checks("ethos_route_topk", q, sub_keys_1, sub_keys_2, out_scores, out_ids)) return rc;
    return hip_status(ethos::launch_route(q, sub_keys_1, sub_keys_2, key_norms, nullptr, n_rows, d_query, n_sub_keys,
                                          top_k, k_cand, dtype, out_scores, out_ids, (hipStream_t)stream),
                      "ethos_route_topk");
}

size_t ethos_route_keys_bytes(int32_t n_sub_keys, int32_t d_query, int32_t dtype) {
    if (!dtype_ok(dtype) || n_sub_keys <= 0 || d_query <= 0 || (d_query & 1) ||
        !ethos::route_supported(n_sub_keys, d_query / 2, dtype))
        return 0;
    return ethos::route_keys_bytes(n_sub_keys, d_query / 2, dtype);
}

int ethos_route_prepare_keys(const void* sub_keys_1, const void* sub_keys_2, int32_t n_sub_keys, int32_t d_query,
                             int32_t dtype, void* prepared, size_t prepared_bytes, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_route_prepare_keys: unknown dtype %d", dtype);
    const size_t need = ethos_route_keys_bytes(n_sub_keys, d_query, dtype);
    if (need == 0)
        return fail(ETHOS_EUNSUPPORTED, "ethos_route_prepare_keys: unsupported sizes K=%d d_query=%d", n_sub_keys,
                    d_query);
    if (!sub_keys_1 || !sub_keys_2 || !prepared) return fail(ETHOS_ENULL, "ethos_route_prepare_keys: null pointer");
    if (prepared_bytes < need)
        return fail(ETHOS_ESIZE, "ethos_route_prepare_keys: prepared holds %zu bytes, needs %zu", prepared_bytes, need);
    if (!aligned16(prepared)) return fail(ETHOS_EALIGN, "ethos_route_prepare_keys: prepared must be 16-byte aligned");
    return hip_status(ethos::launch_route_prepare_keys(sub_keys_1, sub_keys_2, n_sub_keys, d_query, dtype, prepared,
                                                       (hipStream_t)stream),
                      "ethos_route_prepare_keys");
}

int ethos_route_topk_prepared(const void* q, const void* sub_keys_1, const void* sub_keys_2, const float* key_norms,
                              const void* prepared, size_t prepared_bytes, int64_t n_rows, int32_t d_query,
                              int32_t n_sub_keys, int32_t top_k, int32_t k_cand, int32_t dtype, void* out_scores,
                              int32_t* out_ids, void* stream) {
    g_err[0] = 0;
    if (const int rc = route_checks("ethos_route_topk_prepared", n_rows, d_query, n_sub_keys, top_k, k_cand, dtype))
        return rc;
    if (n_rows == 0) return 0;
    if (const int rc = route_prepared_checks("ethos_route_topk_prepared", prepared, prepared_bytes, d_query, n_sub_keys, dtype))
        return rc;
    if (const int rc = route_pointer_checks("ethos_route_topk_prepared", q, sub_keys_1, sub_keys_2, out_scores, out_ids)) return rc;
    return hip_status(ethos::launch_route(q, sub_keys_1, sub_keys_2, key_norms, prepared, n_rows, d_query, n_sub_keys,
                                          top_k, k_cand, dtype, out_scores, out_ids, (hipStream_t)stream),
                      "ethos_route_topk_prepared");
}

size_t ethos_sort_workspace_bytes(int64_t n_pairs, int64_t n_experts) {
    if (n_pairs <= 0 || n_experts <= 0) return 256;
    return ethos::sort_workspace_bytes(n_pairs, n_experts);
}

int ethos_sort_segment(const int32_t* ids, int64_t n_pairs, int64_t n_experts, void* workspace,
                       size_t workspace_bytes, int32_t* perm, int32_t* uniq_ids, int32_t* seg_off,
                       int32_t* pair_slot, int32_t* sorted_slot, int32_t* n_unique, void* stream) {
    g_err[0] = 0;
    if (n_pairs < 0 || n_experts <= 0 || n_experts > INT32_MAX || n_pairs > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_sort_segment: bad sizes n_pairs=%lld n_experts=%lld", (long long)n_pairs,
                    (long long)n_experts);
    if (!seg_off || !n_unique) return fail(ETHOS_ENULL, "ethos_sort_segment: null pointer");
    if (n_pairs == 0)
        return hip_status(ethos::launch_sort_empty(seg_off, n_unique, (hipStream_t)stream), "ethos_sort_segment");
    if (!ids || !workspace || !perm || !uniq_ids || !pair_slot || !sorted_slot)
        return fail(ETHOS_ENULL, "ethos_sort_segment: null pointer");
    if (workspace_bytes < ethos::sort_workspace_bytes(n_pairs, n_experts))
        return fail(ETHOS_EWORKSPACE, "ethos_sort_segment: workspace of %zu bytes, %zu needed", workspace_bytes,
                    ethos::sort_workspace_bytes(n_pairs, n_experts));
    if (!aligned16(workspace)) return fail(ETHOS_EALIGN, "ethos_sort_segment: workspace not 16-byte aligned");
    return hip_status(ethos::launch_sort_segment(ids, n_pairs, n_experts, workspace, perm, uniq_ids, seg_off,
                                                 pair_slot, sorted_slot, n_unique, (hipStream_t)stream),
                      "ethos_sort_segment");
}

int ethos_sort_segment_token_proj(const int32_t* ids, int64_t n_pairs, int64_t n_experts, void* workspace,
                                  size_t workspace_bytes, int32_t* perm, int32_t* uniq_ids, int32_t* seg_off,
                                  int32_t* pair_slot, int32_t* sorted_slot, int32_t* n_unique, const void* x,
                                  const void* w2, const void* wut, int64_t n_tok, int32_t d_model, int32_t d_hidden,
                                  int32_t dtype, void* xp_out, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_sort_segment_token_proj: unknown dtype %d", dtype);
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (n_pairs < 0 || n_experts <= 0 || n_experts > INT32_MAX || n_pairs > INT32_MAX || n_tok < 0 ||
        n_tok > INT32_MAX || d_model <= 0 || d_hidden <= 0)
        return fail(ETHOS_ESIZE, "ethos_sort_segment_token_proj: bad sizes");
    if (d_model % vec || d_hidden % vec)
        return fail(ETHOS_EUNSUPPORTED, "ethos_sort_segment_token_proj: d_model and d_hidden must be multiples of %d",
                    vec);
    if (!seg_off || !n_unique) return fail(ETHOS_ENULL, "ethos_sort_segment_token_proj: null pointer");
    if (n_tok > 0 && (!x || !w2 || !xp_out)) return fail(ETHOS_ENULL, "ethos_sort_segment_token_proj: null pointer");
    if (n_tok > 0 && (!aligned16(x) || !aligned16(w2) || (wut && !aligned16(wut)) || !aligned16(xp_out)))
        return fail(ETHOS_EALIGN, "ethos_sort_segment_token_proj: x, w2, wut and xp_out must be 16-byte aligned");
    if (n_pairs > 0) {
        if (!ids || !perm || !uniq_ids || !pair_slot || !sorted_slot)
            return fail(ETHOS_ENULL, "ethos_sort_segment_token_proj: null pointer");
        if (n_tok > 0 && dtype == ETHOS_BF16) {
            const int rc = ethos::launch_sort_segment_tp(ids, n_pairs, n_experts, perm, uniq_ids, seg_off, pair_slot,
                                                         sorted_slot, n_unique, x, wut, n_tok, d_model, d_hidden,
                                                         xp_out, (hipStream_t)stream);
            if (rc >= 0) return hip_status(rc, "ethos_sort_segment_token_proj");
        }
    }
    // not one launch: the sort, then the projection
    int rc = ethos_sort_segment(ids, n_pairs, n_experts, workspace, workspace_bytes, perm, uniq_ids, seg_off, pair_slot,
                                sorted_slot, n_unique, stream);
    if (rc != 0) return rc;
    return ethos_token_proj(x, w2, wut, n_tok, d_model, d_hidden, dtype, xp_out, stream);
}

int ethos_sort_segment_noalloc(const int32_t* ids, int64_t n_pairs, int64_t n_experts, int32_t* perm,
                               int32_t* uniq_ids, int32_t* seg_off, int32_t* pair_slot, int32_t* sorted_slot,
                               int32_t* n_unique, void* stream) {
    g_err[0] = 0;
    if (n_pairs < 0 || n_experts <= 0 || n_experts > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_sort_segment_noalloc: bad sizes n_pairs=%lld n_experts=%lld",
                    (long long)n_pairs, (long long)n_experts);
    if (n_pairs > ETHOS_NOALLOC_MAX_PAIRS)
        return fail(ETHOS_ESIZE,
                    "ethos_sort_segment_noalloc: %lld pairs exceed the %d its static workspace holds; use "
                    "ethos_sort_segment with a caller workspace", (long long)n_pairs, ETHOS_NOALLOC_MAX_PAIRS);
    if (!seg_off || !n_unique) return fail(ETHOS_ENULL, "ethos_sort_segment_noalloc: null pointer");
    if (n_pairs == 0)
        return hip_status(ethos::launch_sort_empty(seg_off, n_unique, (hipStream_t)stream),
                          "ethos_sort_segment_noalloc");
    if (!ids || !perm || !uniq_ids || !pair_slot || !sorted_slot)
        return fail(ETHOS_ENULL, "ethos_sort_segment_noalloc: null pointer");
    if (ethos::sort_workspace_bytes(n_pairs, n_experts) > sizeof(scratch))
        return fail(ETHOS_EWORKSPACE, "ethos_sort_segment_noalloc: static workspace sizing");
    int rc = 0;
    void* ws = scratch_ptr(&rc);
    if (!ws) return rc;
    return hip_status(ethos::launch_sort_segment(ids, n_pairs, n_experts, ws, perm, uniq_ids, seg_off, pair_slot,
                                                 sorted_slot, n_unique, (hipStream_t)stream),
                      "ethos_sort_segment_noalloc");
}

int ethos_generate(const void* latents, int64_t n_experts, const int32_t* uniq_ids, const int32_t* n_unique,
                   int64_t max_unique, const void* w1, const void* w2, int32_t d_latent, int32_t d_hidden,
                   int32_t d_model, int32_t dtype, void* h_out, void* v_out, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_generate: unknown dtype %d", dtype);
    if (n_experts <= 0 || max_unique < 0 || d_latent <= 0 || d_hidden <= 0 || d_model <= 0)
        return fail(ETHOS_ESIZE, "ethos_generate: bad sizes");
    const int kq = dtype == ETHOS_BF16 ? 16 : 2;
    if (d_latent % kq || d_hidden % 32 || d_model % 32)
        return fail(ETHOS_EUNSUPPORTED,
                    "ethos_generate: needs d_latent %% %d == 0, d_hidden %% 32 == 0, d_model %% 32 == 0 "
                    "(got %d, %d, %d)", kq, d_latent, d_hidden, d_model);
    if (ethos::generate_smem_bytes(d_latent, d_hidden, dtype) > 160 * 1024)
        return fail(ETHOS_EUNSUPPORTED, "ethos_generate: d_latent + d_hidden too large for LDS");
    if (max_unique == 0) return 0;
    // v_out == NULL: hidden rows only (w2 is then not read)
    if (!latents || !uniq_ids || !n_unique || !w1 || !h_out || (v_out && !w2))
        return fail(ETHOS_ENULL, "ethos_generate: null pointer");
    if (dtype == ETHOS_BF16 &&
        (!aligned16(w1) || (v_out && !aligned16(w2)) || !aligned16(h_out) || (v_out && !aligned16(v_out))))
        return fail(ETHOS_EALIGN, "ethos_generate: weights and outputs must be 16-byte aligned");
    return hip_status(ethos::launch_generate(latents, n_experts, uniq_ids, n_unique, max_unique, w1, w2, d_latent,
                                             d_hidden, d_model, dtype, h_out, v_out, num_cus(), (hipStream_t)stream),
                      "ethos_generate");
}

size_t ethos_apply_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_hidden, int32_t dtype) {
    if (n_tok <= 0 || n_heads <= 0 || top_k <= 0 || d_hidden <= 0) return 256;
    return ethos::apply_workspace_bytes(n_tok, n_heads, top_k, d_hidden, dtype);
}

int ethos_apply_scatter(const void* x, const void* w2, const void* h, const void* v, const int32_t* perm,
                        const int32_t* sorted_slot, const int32_t* pair_slot, const void* scores, int64_t n_tok,
                        int32_t n_heads, int32_t top_k, int32_t d_model, int32_t d_hidden, int32_t dtype,
                        void* workspace, size_t workspace_bytes, void* out, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_apply_scatter: unknown dtype %d", dtype);
    if (n_tok < 0 || n_heads <= 0 || top_k <= 0 || d_model <= 0 || d_hidden <= 0)
        return fail(ETHOS_ESIZE, "ethos_apply_scatter: bad sizes");
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (d_model % vec || d_hidden % vec || ethos::apply_chunks(d_model, dtype) > 8 ||
        ethos::apply_chunks(d_hidden, dtype) > 8)
        return fail(ETHOS_EUNSUPPORTED,
                    "ethos_apply_scatter: d_model=%d and d_hidden=%d must be multiples of %d and <= %d", d_model,
                    d_hidden, vec, 8 * 64 * vec);
    if (n_tok * n_heads * top_k > INT32_MAX || n_tok > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_apply_scatter: too many pairs");
    if (n_tok == 0) return 0;
    if (!x || !w2 || !h || !v || !perm || !sorted_slot || !pair_slot || !scores || !workspace || !out)
        return fail(ETHOS_ENULL, "ethos_apply_scatter: null pointer");
    const size_t need = ethos::apply_workspace_bytes(n_tok, n_heads, top_k, d_hidden, dtype);
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_apply_scatter: workspace of %zu bytes, %zu needed", workspace_bytes,
                    need);
    if (!aligned16(x) || !aligned16(w2) || !aligned16(h) || !aligned16(v) || !aligned16(workspace) ||
        !aligned16(out))
        return fail(ETHOS_EALIGN, "ethos_apply_scatter: x, w2, h, v, workspace and out must be 16-byte aligned");
    return hip_status(ethos::launch_apply(x, w2, h, v, perm, sorted_slot, pair_slot, scores, n_tok, n_heads, top_k,
                                          d_model, d_hidden, dtype, workspace, out, num_cus(), (hipStream_t)stream),
                      "ethos_apply_scatter");
}

size_t ethos_apply_hidden_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_model,
                                          int32_t d_hidden, int32_t dtype) {
    if (n_tok <= 0 || n_heads <= 0 || top_k <= 0 || d_model <= 0 || d_hidden <= 0) return 256;
    return ethos::apply_hidden_workspace_bytes(n_tok, n_heads, top_k, d_model, d_hidden, dtype);
}

int ethos_apply_hidden(const void* x, const void* w2, const void* h, const int32_t* perm, const int32_t* sorted_slot,
                       const int32_t* pair_slot, const void* scores, int64_t n_tok, int32_t n_heads, int32_t top_k,
                       int32_t d_model, int32_t d_hidden, int32_t dtype, void* workspace, size_t workspace_bytes,
                       void* out, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_apply_hidden: unknown dtype %d", dtype);
    if (n_tok < 0 || n_heads <= 0 || top_k <= 0 || d_model <= 0 || d_hidden <= 0)
        return fail(ETHOS_ESIZE, "ethos_apply_hidden: bad sizes");
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (d_model % vec || d_hidden % vec || d_model > 4096 || ethos::apply_chunks(d_hidden, dtype) > 8)
        return fail(ETHOS_EUNSUPPORTED,
                    "ethos_apply_hidden: d_model=%d and d_hidden=%d must be multiples of %d, d_model <= 4096, "
                    "d_hidden <= %d", d_model, d_hidden, vec, 8 * 64 * vec);
    if (n_tok * n_heads * top_k > INT32_MAX || n_tok > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_apply_hidden: too many pairs");
    if (n_tok == 0) return 0;
    if (!x || !w2 || !h || !perm || !sorted_slot || !pair_slot || !scores || !workspace || !out)
        return fail(ETHOS_ENULL, "ethos_apply_hidden: null pointer");
    const size_t need = ethos::apply_hidden_workspace_bytes(n_tok, n_heads, top_k, d_model, d_hidden, dtype);
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_apply_hidden: workspace of %zu bytes, %zu needed", workspace_bytes,
                    need);
    if (!aligned16(x) || !aligned16(w2) || !aligned16(h) || !aligned16(workspace) || !aligned16(out))
        return fail(ETHOS_EALIGN, "ethos_apply_hidden: x, w2, h, workspace and out must be 16-byte aligned");
    const int rc = ethos::launch_apply_hidden(x, w2, h, perm, sorted_slot, pair_slot, scores, n_tok, n_heads, top_k,
                                              d_model, d_hidden, dtype, workspace, out, num_cus(), (hipStream_t)stream);
    if (rc < 0) return fail(ETHOS_EUNSUPPORTED, "ethos_apply_hidden: d_hidden=%d not supported", d_hidden);
    return hip_status(rc, "ethos_apply_hidden");
}

size_t ethos_expert_forward_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t top_k, int64_t max_unique,
                                            int32_t d_model, int32_t d_hidden, int32_t dtype, int32_t order) {
    if (n_tok <= 0 || n_heads <= 0 || top_k <= 0 || max_unique < 0 || d_model <= 0 || d_hidden <= 0 ||
        (order != 0 && order != 1))
        return 256;
    return ethos::expert_forward_workspace_bytes(n_tok, n_heads, top_k, max_unique, d_model, d_hidden, dtype, order);
}

int ethos_token_proj(const void* x, const void* w2, const void* wut, int64_t n_tok, int32_t d_model,
                     int32_t d_hidden, int32_t dtype, void* xp_out, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_token_proj: unknown dtype %d", dtype);
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (n_tok < 0 || d_model <= 0 || d_hidden <= 0 || n_tok > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_token_proj: bad sizes");
    if (d_model % vec || d_hidden % vec)
        return fail(ETHOS_EUNSUPPORTED, "ethos_token_proj: d_model and d_hidden must be multiples of %d", vec);
    if (n_tok == 0) return 0;
    if (!x || !w2 || !xp_out) return fail(ETHOS_ENULL, "ethos_token_proj: null pointer");
    if (!aligned16(x) || !aligned16(w2) || (wut && !aligned16(wut)) || !aligned16(xp_out))
        return fail(ETHOS_EALIGN, "ethos_token_proj: x, w2, wut and xp_out must be 16-byte aligned");
    const int rc = ethos::launch_token_proj_out(x, w2, dtype == ETHOS_BF16 ? wut : nullptr, n_tok, d_model, d_hidden,
                                                dtype, xp_out, num_cus(), (hipStream_t)stream);
    if (rc < 0) return fail(ETHOS_ENULL, "ethos_token_proj: bf16 needs wut (W_u^T)");
    return hip_status(rc, "ethos_token_proj");
}

static int expert_forward_checks(const char* name, const void* x, const void* latents, int64_t n_experts, const void* w1, const void* w2,
                                 const void* wut, const void* xp, const int32_t* uniq_ids, const int32_t* seg_off,
                                 const int32_t* n_unique, int64_t max_unique,
                                 const int32_t* perm, const int32_t* sorted_slot, const int32_t* pair_slot, const void* scores,
                                 int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_latent, int32_t d_hidden,
                                 int32_t d_model, int32_t dtype, int32_t order, const void* workspace, size_t workspace_bytes,
                                 const void* h_out, const void* out) {
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "%s: unknown dtype %d", name, dtype);
    if (order != 0 && order != 1) return fail(ETHOS_ESIZE, "%s: order must be 0 or 1, got %d", name, order);
    if (n_tok < 0 || n_heads <= 0 || top_k <= 0 || n_experts <= 0 || max_unique < 0 || d_latent <= 0 ||
        d_hidden <= 0 || d_model <= 0)
        return fail(ETHOS_ESIZE, "%s: bad sizes", name);
    if (n_tok * n_heads * top_k > INT32_MAX || n_tok > INT32_MAX)
        return fail(ETHOS_ESIZE, "%s: too many pairs", name);
    const int kq = dtype == ETHOS_BF16 ? 16 : 2;
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (d_latent % kq || d_hidden % 32 || d_model % 32 || d_model > 4096 ||
        ethos::apply_chunks(d_model, dtype) > 8 || ethos::apply_chunks(d_hidden, dtype) > 8 ||
        ethos::generate_smem_bytes(d_latent, d_hidden, dtype) > 160 * 1024 || d_model % vec || d_hidden % vec)
        return fail(ETHOS_EUNSUPPORTED,
                    "%s: needs d_latent %% %d == 0, d_hidden and d_model multiples of 32 with "
                    "d_model <= 4096 and d_hidden <= %d (got %d, %d, %d)", name, kq, 8 * 64 * vec, d_latent, d_hidden,
                    d_model);
    if (n_tok == 0) return 0;
    if (max_unique < 1) return fail(ETHOS_ESIZE, "%s: max_unique must be >= 1 for a nonempty batch", name);
    if (!x || !latents || !w1 || !w2 || !uniq_ids || !seg_off || !n_unique || !perm || !sorted_slot || !pair_slot ||
        !scores || !workspace || !h_out || !out)
        return fail(ETHOS_ENULL, "%s: null pointer", name);
    const size_t need = ethos::expert_forward_workspace_bytes(n_tok, n_heads, top_k, max_unique, d_model, d_hidden,
                                                              dtype, order);
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "%s: workspace of %zu bytes, %zu needed", name, workspace_bytes, need);
    if (!aligned16(x) || !aligned16(w1) || !aligned16(w2) || (wut && !aligned16(wut)) || (xp && !aligned16(xp)) ||
        !aligned16(workspace) || !aligned16(h_out) || !aligned16(out))
        return fail(ETHOS_EALIGN, "%s: x, w1, w2, wut, xp, workspace, h_out and out must be 16-byte aligned", name);
    return 0;
}

int ethos_expert_forward(const void* x, const void* latents, int64_t n_experts, const void* w1, const void* w2,
                         const void* wut, const void* xp, const int32_t* uniq_ids, const int32_t* seg_off,
                         const int32_t* n_unique, int64_t max_unique,
                         const int32_t* perm, const int32_t* sorted_slot, const int32_t* pair_slot, const void* scores,
                         int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_latent, int32_t d_hidden,
                         int32_t d_model, int32_t dtype, int32_t order, void* workspace, size_t workspace_bytes,
                         void* h_out, void* out, void* stream) {
    g_err[0] = 0;
    if (const int rc = expert_forward_checks("ethos_expert_forward", x, latents, n_experts, w1, w2, wut, xp, uniq_ids, seg_off, n_unique,
                                             max_unique, perm, sorted_slot, pair_slot, scores, n_tok, n_heads, top_k, d_latent,
                                             d_hidden, d_model, dtype, order, workspace, workspace_bytes, h_out, out))
        return rc;
    if (n_tok == 0) return 0;
    const int rc = ethos::launch_expert_forward(x, latents, n_experts, w1, w2, dtype == ETHOS_BF16 ? wut : nullptr,
                                                xp, uniq_ids, seg_off, n_unique, max_unique, perm, sorted_slot,
                                                pair_slot, scores,
                                                n_tok, n_heads, top_k, d_latent, d_hidden, d_model, dtype, order,
                                                workspace, h_out, out, num_cus(), (hipStream_t)stream);
    if (rc < 0) return fail(ETHOS_EUNSUPPORTED, "ethos_expert_forward: shape not supported");
    return hip_status(rc, "ethos_expert_forward");
}

size_t ethos_expert_backward_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_hidden) {
    if (n_tok < 0 || n_heads <= 0 || top_k <= 0 || d_hidden <= 0) return 0;
    return ethos::expert_backward_workspace_bytes(n_tok * n_heads * top_k, d_hidden);
}

int ethos_expert_backward(const void* h, const float* xp, const float* dyb, const int32_t* pair_slot,
                          const int32_t* perm, const int32_t* sorted_slot, const int32_t* seg_off, const void* scores,
                          int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_hidden, int32_t dtype,
                          void* workspace, size_t workspace_bytes, float* dscores, float* hacc, float* dxp, float* dh,
                          void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_expert_backward: unknown dtype %d", dtype);
    if (n_tok < 0 || n_heads <= 0 || top_k <= 0 || d_hidden <= 0)
        return fail(ETHOS_ESIZE, "ethos_expert_backward: bad sizes");
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (d_hidden % vec || ethos::apply_chunks(d_hidden, dtype) > 8)
        return fail(ETHOS_EUNSUPPORTED, "ethos_expert_backward: d_hidden=%d must be a multiple of %d and <= %d",
                    d_hidden, vec, 8 * 64 * vec);
    if (n_tok * n_heads * top_k > INT32_MAX || n_tok > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_expert_backward: too many pairs");
    if (n_tok == 0) return 0;
    if (!h || !xp || !dyb || !pair_slot || !perm || !sorted_slot || !seg_off || !scores || !workspace || !dscores ||
        !hacc || !dxp || !dh)
        return fail(ETHOS_ENULL, "ethos_expert_backward: null pointer");
    const size_t need = ethos::expert_backward_workspace_bytes(n_tok * n_heads * top_k, d_hidden);
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_expert_backward: workspace of %zu bytes, %zu needed", workspace_bytes,
                    need);
    if (!aligned16(h) || !aligned16(workspace))
        return fail(ETHOS_EALIGN, "ethos_expert_backward: h and workspace must be 16-byte aligned");
    const int rc = ethos::launch_expert_backward(h, xp, dyb, pair_slot, perm, sorted_slot, seg_off, scores, n_tok,
                                                 n_heads, top_k, d_hidden, dtype, workspace, dscores, hacc, dxp, dh,
                                                 num_cus(), (hipStream_t)stream);
    if (rc < 0) return fail(ETHOS_EUNSUPPORTED, "ethos_expert_backward: d_hidden=%d not supported", d_hidden);
    return hip_status(rc, "ethos_expert_backward");
}

size_t ethos_expert_grads_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t top_k, int64_t max_unique,
                                          int32_t d_latent, int32_t d_hidden, int32_t d_model) {
    if (n_tok <= 0 || n_heads <= 0 || top_k <= 0 || max_unique <= 0 || d_latent <= 0 || d_hidden <= 0 || d_model <= 0) return 256;
    return ethos::expert_grads_workspace_bytes(n_tok, n_heads, top_k, max_unique, d_latent, d_hidden, d_model, num_cus());
}

int ethos_expert_grads(const void* x, const void* dy, const void* h, const void* latents, const void* w1, const void* w2,
                       const int32_t* uniq_ids, const int32_t* seg_off, const int32_t* n_unique, int64_t max_unique,
                       const int32_t* perm, const int32_t* sorted_slot, const int32_t* pair_slot, const void* scores,
                       int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_latent, int32_t d_hidden, int32_t d_model,
                       int32_t dtype, void* workspace, size_t workspace_bytes, void* dx, float* dscores, void* dlatents,
                       void* dw1, void* dw2, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_expert_grads: unknown dtype %d", dtype);
    if (n_tok < 0 || n_heads <= 0 || top_k <= 0 || max_unique < 0 || d_latent <= 0 || d_hidden <= 0 || d_model <= 0)
        return fail(ETHOS_ESIZE, "ethos_expert_grads: bad sizes");
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (d_latent % 8 || d_hidden % 8 || d_model % 8 || ethos::apply_chunks(d_hidden, dtype) > 8)
        return fail(ETHOS_EUNSUPPORTED,
                    "ethos_expert_grads: d_latent=%d, d_hidden=%d and d_model=%d must be multiples of 8, d_hidden <= %d",
                    d_latent, d_hidden, d_model, 8 * 64 * vec);
    if (n_tok > INT32_MAX || n_tok * n_heads * top_k > INT32_MAX || max_unique > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_expert_grads: too many pairs");
    if (n_tok == 0) return 0;
    if (max_unique < 1) return fail(ETHOS_ESIZE, "ethos_expert_grads: max_unique must be >= 1 for a nonempty batch");
    if (!x || !dy || !h || !latents || !w1 || !w2 || !uniq_ids || !seg_off || !n_unique || !perm || !sorted_slot || !pair_slot ||
        !scores || !workspace || !dx || !dscores || !dlatents || !dw1 || !dw2)
        return fail(ETHOS_ENULL, "ethos_expert_grads: null pointer");
    const size_t need = ethos::expert_grads_workspace_bytes(n_tok, n_heads, top_k, max_unique, d_latent, d_hidden, d_model,
                                                            num_cus());
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_expert_grads: workspace of %zu bytes, %zu needed", workspace_bytes, need);
    if (!aligned16(x) || !aligned16(dy) || !aligned16(h) || !aligned16(latents) || !aligned16(w1) || !aligned16(w2) ||
        !aligned16(workspace))
        return fail(ETHOS_EALIGN, "ethos_expert_grads: x, dy, h, latents, w1, w2 and workspace must be 16-byte aligned");
    const int rc = ethos::launch_expert_grads(x, dy, h, latents, w1, w2, uniq_ids, seg_off, n_unique, max_unique, perm,
                                              sorted_slot, pair_slot, scores, n_tok, n_heads, top_k, d_latent, d_hidden,
                                              d_model, dtype, workspace, dx, dscores, dlatents, dw1, dw2, num_cus(),
                                              (hipStream_t)stream);
    if (rc < 0) return fail(ETHOS_EUNSUPPORTED, "ethos_expert_grads: d_hidden=%d not supported", d_hidden);
    return hip_status(rc, "ethos_expert_grads");
}

size_t ethos_query_bn_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t d_query) {
    if (n_tok <= 0 || n_heads <= 0 || d_query <= 0) return 256;
    return ethos::query_bn_workspace_bytes(n_tok, n_heads, d_query);
}

int ethos_query_bn_train(const void* v, int64_t n_tok, int32_t n_heads, int32_t d_query, int32_t dtype, const void* const* gamma,
                         const void* const* beta, void* const* running_mean, void* const* running_var,
                         const float* const* batch_mean, const float* const* batch_var, double momentum, double eps,
                         void* workspace, size_t workspace_bytes, void* q, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_query_bn_train: unknown dtype %d", dtype);
    if (n_tok < 2 || n_tok > INT32_MAX || n_heads <= 0 || d_query <= 0)
        return fail(ETHOS_ESIZE, "ethos_query_bn_train: bad sizes (batch statistics need two tokens)");
    if (n_heads > ethos::kMaxBnHeads || d_query % 4)
        return fail(ETHOS_EUNSUPPORTED, "ethos_query_bn_train: at most %d heads and d_query %% 4 == 0", ethos::kMaxBnHeads);
    if (!v || !gamma || !beta || (!running_mean) != (!running_var) || (!batch_mean) != (!batch_var) || !workspace ||
        !q)
        return fail(ETHOS_ENULL, "ethos_query_bn_train: null pointer");
    for (int h = 0; h < n_heads; ++h)
        if (!gamma[h] || !beta[h] || (running_mean && (!running_mean[h] || !running_var[h])) ||
            (batch_mean && (!batch_mean[h] || !batch_var[h])))
            return fail(ETHOS_ENULL, "ethos_query_bn_train: null pointer (head %d)", h);
    const size_t need = ethos::query_bn_workspace_bytes(n_tok, n_heads, d_query);
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_query_bn_train: workspace of %zu bytes, %zu needed", workspace_bytes, need);
    if (!aligned16(v) || !aligned16(workspace) || !aligned16(q))
        return fail(ETHOS_EALIGN, "ethos_query_bn_train: v, workspace and q must be 16-byte aligned");
    return hip_status(ethos::launch_query_bn(v, n_tok, n_heads, d_query, dtype, gamma, beta, running_mean, running_var, batch_mean,
                                             batch_var, momentum, eps, workspace, q, num_cus(), (hipStream_t)stream),
                      "ethos_query_bn_train");
}

int ethos_bn_coefficients(int32_t n_heads, int32_t d_query, int32_t dtype, const void* const* gamma, const void* const* beta,
                          const void* const* running_mean, const void* const* running_var, double eps, float* alpha_out,
                          float* beta_out, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_bn_coefficients: unknown dtype %d", dtype);
    if (n_heads <= 0 || d_query <= 0) return fail(ETHOS_ESIZE, "ethos_bn_coefficients: bad sizes");
    if (n_heads > ethos::kMaxBnHeads)
        return fail(ETHOS_EUNSUPPORTED, "ethos_bn_coefficients: at most %d heads", ethos::kMaxBnHeads);
    if (!alpha_out || !beta_out) return fail(ETHOS_ENULL, "ethos_bn_coefficients: null pointer");
    return hip_status(ethos::launch_bn_coefficients(n_heads, d_query, dtype, gamma, beta, (void* const*)running_mean,
                                                    (void* const*)running_var, eps, alpha_out, beta_out, (hipStream_t)stream),
                      "ethos_bn_coefficients");
}

size_t ethos_gate_grads_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_model, int32_t d_query,
                                        int32_t n_sub) {
    if (n_tok <= 0 || n_heads <= 0 || top_k <= 0 || d_model <= 0 || d_query <= 0 || n_sub <= 0) return 256;
    return ethos::gate_grads_workspace_bytes(n_tok, n_heads, top_k, d_model, d_query, n_sub, num_cus());
}

int ethos_gate_grads(const void* x, const int32_t* ids, const float* dscores, const void* wq, const void* bq,
                     const void* sub_keys_1, const void* sub_keys_2, const void* const* gamma, const void* const* beta,
                     const void* const* running_mean, const void* const* running_var, double eps, int64_t n_tok, int32_t d_model,
                     int32_t n_heads, int32_t d_query, int32_t n_sub, int32_t top_k, int32_t dtype, void* workspace,
                     size_t workspace_bytes, void* dx, void* dwq, void* dbq, void* dgamma, void* dbeta, void* dkeys_1,
                     void* dkeys_2, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_gate_grads: unknown dtype %d", dtype);
    if (n_tok < 0 || n_heads <= 0 || d_query <= 0 || n_sub <= 0 || top_k <= 0 || d_model <= 0)
        return fail(ETHOS_ESIZE, "ethos_gate_grads: bad sizes");
    if (d_model % 8 || !ethos::gate_grads_supported(n_heads, d_query, n_sub, top_k))
        return fail(ETHOS_EUNSUPPORTED,
                    "ethos_gate_grads: needs d_model %% 8 == 0, d_query %% 8 == 0 and at most 512 with whole lanes, at most %d "
                    "heads, 1024 sub-keys and top_k 64 (got d_model %d, d_query %d, %d heads, %d, %d)",
                    ethos::kMaxBnHeads, d_model, d_query, n_heads, n_sub, top_k);
    if (n_tok > INT32_MAX || n_tok * n_heads * top_k > INT32_MAX) return fail(ETHOS_ESIZE, "ethos_gate_grads: too many pairs");
    if (n_tok == 0) return 0;
    if (!x || !ids || !dscores || !wq || !bq || !sub_keys_1 || !sub_keys_2 || !gamma || !beta || (!running_mean) != (!running_var) ||
        !workspace || !dbq || !dgamma || !dbeta || !dkeys_1 || !dkeys_2)
        return fail(ETHOS_ENULL, "ethos_gate_grads: null pointer");
    for (int h = 0; h < n_heads; ++h)
        if (!gamma[h] || !beta[h] || (running_mean && (!running_mean[h] || !running_var[h])))
            return fail(ETHOS_ENULL, "ethos_gate_grads: null pointer (head %d)", h);
    const size_t need = ethos::gate_grads_workspace_bytes(n_tok, n_heads, top_k, d_model, d_query, n_sub, num_cus());
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_gate_grads: workspace of %zu bytes, %zu needed", workspace_bytes, need);
    if (!aligned16(x) || !aligned16(wq) || !aligned16(sub_keys_1) || !aligned16(sub_keys_2) || !aligned16(workspace))
        return fail(ETHOS_EALIGN, "ethos_gate_grads: x, wq, the sub-keys and workspace must be 16-byte aligned");
    return hip_status(ethos::launch_gate_grads(x, ids, dscores, wq, bq, sub_keys_1, sub_keys_2, gamma, beta,
                                               (void* const*)running_mean, (void* const*)running_var, eps, n_tok, d_model, n_heads,
                                               d_query, n_sub, top_k, dtype, workspace, dx, dwq, dbq, dgamma, dbeta, dkeys_1,
                                               dkeys_2, num_cus(), (hipStream_t)stream),
                      "ethos_gate_grads");
}

int ethos_rms_norm(const void* x, int64_t ldx, const void* weight, int64_t rows, int32_t d, float eps, int32_t dtype, void* y,
                   void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_rms_norm: unknown dtype %d", dtype);
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (rows < 0 || rows > INT32_MAX || d <= 0 || ldx < d) return fail(ETHOS_ESIZE, "ethos_rms_norm: bad sizes");
    if (d % vec || ldx % vec || d > 512 * vec)
        return fail(ETHOS_EUNSUPPORTED, "ethos_rms_norm: d and ldx must be multiples of %d, d <= %d", vec, 512 * vec);
    if (rows == 0) return 0;
    if (!x || !weight || !y) return fail(ETHOS_ENULL, "ethos_rms_norm: null pointer");
    if (!aligned16(x) || !aligned16(weight) || !aligned16(y))
        return fail(ETHOS_EALIGN, "ethos_rms_norm: x, weight and y must be 16-byte aligned");
    return hip_status(ethos::launch_rms_norm(x, ldx, weight, rows, d, eps, dtype, y, (hipStream_t)stream), "ethos_rms_norm");
}

int ethos_swiglu(const void* gate_up, int64_t rows, int32_t d, int32_t dtype, void* out, void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_swiglu: unknown dtype %d", dtype);
    const int vec = dtype == ETHOS_BF16 ? 8 : 4;
    if (rows < 0 || d <= 0) return fail(ETHOS_ESIZE, "ethos_swiglu: bad sizes");
    if (d % vec) return fail(ETHOS_EUNSUPPORTED, "ethos_swiglu: d must be a multiple of %d", vec);
    if (rows == 0) return 0;
    if (!gate_up || !out) return fail(ETHOS_ENULL, "ethos_swiglu: null pointer");
    if (!aligned16(gate_up) || !aligned16(out)) return fail(ETHOS_EALIGN, "ethos_swiglu: gate_up and out must be 16-byte aligned");
    return hip_status(ethos::launch_swiglu(gate_up, rows, d, dtype, out, num_cus(), (hipStream_t)stream), "ethos_swiglu");
}

size_t ethos_mla_attention_workspace_bytes(int64_t n_seq, int64_t seq_len) {
    if (n_seq <= 0 || seq_len <= 0) return 256;
    return ethos::mla_attention_workspace_bytes(n_seq, seq_len);
}

int ethos_mla_attention(const void* q, const void* kv, const void* k_rot, int64_t k_rot_ld, const int64_t* positions,
                        const float* rates, int64_t n_seq, int64_t seq_len, int32_t n_heads, int32_t nope, int32_t rope, int32_t v_dim,
                        int32_t dtype, float scale, void* workspace, size_t workspace_bytes, void* out, void* stream) {
    g_err[0] = 0;
    if (dtype != ETHOS_BF16) return fail(ETHOS_EDTYPE, "ethos_mla_attention: bf16 only, got dtype %d", dtype);
    if (n_seq < 0 || seq_len < 0 || n_heads <= 0 || k_rot_ld < rope) return fail(ETHOS_ESIZE, "ethos_mla_attention: bad sizes");
    if (!ethos::mla_attention_supported(nope, rope, v_dim) || k_rot_ld % 2)
        return fail(ETHOS_EUNSUPPORTED, "ethos_mla_attention: needs widths 64, 64, 64 (got %d, %d, %d) and an even k_rot_ld", nope,
                    rope, v_dim);
    if (n_seq * n_heads > INT32_MAX / 2 || seq_len > INT32_MAX / 2 ||
        n_seq * n_heads * ((seq_len + 63) / 64) > INT32_MAX / 2 || n_seq * seq_len > INT32_MAX)
        return fail(ETHOS_ESIZE, "ethos_mla_attention: too many rows");
    if (n_seq == 0 || seq_len == 0) return 0;
    if (!q || !kv || !k_rot || !positions || !rates || !workspace || !out)
        return fail(ETHOS_ENULL, "ethos_mla_attention: null pointer");
    const size_t need = ethos::mla_attention_workspace_bytes(n_seq, seq_len);
    if (workspace_bytes < need)
        return fail(ETHOS_EWORKSPACE, "ethos_mla_attention: workspace of %zu bytes, %zu needed", workspace_bytes, need);
    if (!aligned16(q) || !aligned16(kv) || !aligned16(workspace) || !aligned16(out) || ((uintptr_t)k_rot & 3u))
        return fail(ETHOS_EALIGN, "ethos_mla_attention: q, kv, workspace and out must be 16-byte, k_rot 4-byte aligned");
    return hip_status(ethos::launch_mla_attention(q, kv, k_rot, k_rot_ld, positions, rates, n_seq, seq_len, n_heads, scale, workspace,
                                                  out, num_cus(), (hipStream_t)stream),
                      "ethos_mla_attention");
}

namespace {

// ethos_layer_forward's workspace: what lives to the end, then one region that the projection (its
// scratch and the queries), the sort and the expert stages use in turn.
struct LayerLayout {
    size_t gates, ids, perm, pair_slot, sorted_slot, uniq, seg_off, n_unique, xp, shared, q, qws, h, ews, total;
    size_t qws_bytes, sort_bytes, ews_bytes;
    int64_t n_pairs, max_u;
};

LayerLayout layer_layout(int64_t n_tok, int H, int k, int d, int dq, int64_t n_experts, int dh, int dtype, int order) {
    LayerLayout l{};
    const size_t eb = dtype == ETHOS_BF16 ? 2 : 4;
    l.n_pairs = n_tok * H * k;
    l.max_u = l.n_pairs < n_experts ? l.n_pairs : n_experts;
    l.max_u = l.max_u < 1 ? 1 : l.max_u;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t r = at;
        at += (bytes + 255) & ~(size_t)255;
        return r;
    };
    l.gates = take((size_t)l.n_pairs * eb);
    l.ids = take((size_t)l.n_pairs * 4);
    l.perm = take((size_t)l.n_pairs * 4);
    l.pair_slot = take((size_t)l.n_pairs * 4);
    l.sorted_slot = take((size_t)l.n_pairs * 4);
    l.uniq = take((size_t)l.max_u * 4);
    l.seg_off = take((size_t)(l.max_u + 1) * 4);
    l.n_unique = take(4);
    l.xp = take((size_t)n_tok * dh * eb);
    l.shared = at;
    l.qws_bytes = ethos_query_proj_workspace_bytes(n_tok, d, H, dq, dtype);
    l.q = take((size_t)n_tok * H * dq * eb);
    l.qws = take(l.qws_bytes);
    l.total = at;
    l.sort_bytes = ethos_sort_workspace_bytes(l.n_pairs, n_experts);
    at = l.shared;
    take(l.sort_bytes);
    l.total = l.total > at ? l.total : at;
    at = l.shared;
    l.ews_bytes = ethos_expert_forward_workspace_bytes(n_tok, H, k, l.max_u, d, dh, dtype, order);
    l.h = take((size_t)l.max_u * dh * eb);
    l.ews = take(l.ews_bytes);
    l.total = l.total > at ? l.total : at;
    return l;
}

bool layer_sizes_ok(int64_t n_tok, int H, int k, int d, int dq, int64_t n_experts, int dh) {
    return n_tok > 0 && n_tok <= INT32_MAX && H > 0 && k > 0 && d > 0 && dq > 0 && n_experts > 0 && dh > 0 &&
           n_tok <= INT32_MAX / H / k;
}

}  // namespace

size_t ethos_layer_forward_workspace_bytes(int64_t n_tok, int32_t n_heads, int32_t top_k, int32_t d_model, int32_t d_query,
                                           int64_t n_experts, int32_t d_hidden, int32_t dtype, int32_t order) {
    if (!layer_sizes_ok(n_tok, n_heads, top_k, d_model, d_query, n_experts, d_hidden)) return 256;
    return layer_layout(n_tok, n_heads, top_k, d_model, d_query, n_experts, d_hidden, dtype, order).total;
}

int ethos_layer_forward(const void* x, const void* wq, const void* wq_prepared, size_t wq_prepared_bytes, const void* bq,
                        const float* bn_alpha, const float* bn_beta, const void* sub_keys_1, const void* sub_keys_2,
                        const float* key_norms, const void* keys_prepared, size_t keys_prepared_bytes, const void* latents,
                        const void* w1, const void* w2, const void* wut, int64_t n_tok, int32_t d_model, int32_t n_heads,
                        int32_t d_query, int32_t n_sub_keys, int32_t top_k, int32_t k_cand, int64_t n_experts, int32_t d_latent,
                        int32_t d_hidden, int32_t dtype, int32_t order, void* workspace, size_t workspace_bytes, void* out,
                        void* stream) {
    g_err[0] = 0;
    if (!dtype_ok(dtype)) return fail(ETHOS_EDTYPE, "ethos_layer_forward: unknown dtype %d", dtype);
    if (order != 0 && order != 1) return fail(ETHOS_ESIZE, "ethos_layer_forward: order must be 0 or 1, got %d", order);
    if (n_tok == 0) return 0;
    if (!layer_sizes_ok(n_tok, n_heads, top_k, d_model, d_query, n_experts, d_hidden) || d_latent <= 0)
        return fail(ETHOS_ESIZE, "ethos_layer_forward: bad sizes");
    if (!workspace) return fail(ETHOS_ENULL, "ethos_layer_forward: null pointer");
    if (!aligned16(workspace)) return fail(ETHOS_EALIGN, "ethos_layer_forward: workspace must be 16-byte aligned");
    const LayerLayout l = layer_layout(n_tok, n_heads, top_k, d_model, d_query, n_experts, d_hidden, dtype, order);
    if (workspace_bytes < l.total)
        return fail(ETHOS_EWORKSPACE, "ethos_layer_forward: workspace of %zu bytes, %zu needed", workspace_bytes, l.total);
    unsigned char* w = static_cast<unsigned char*>(workspace);
    void *q = w + l.q, *gates = w + l.gates, *xp = nullptr;
    int32_t *ids = (int32_t*)(w + l.ids), *perm = (int32_t*)(w + l.perm), *uniq = (int32_t*)(w + l.uniq);
    int32_t *seg_off = (int32_t*)(w + l.seg_off), *pair_slot = (int32_t*)(w + l.pair_slot);
    int32_t *sorted_slot = (int32_t*)(w + l.sorted_slot), *n_unique = (int32_t*)(w + l.n_unique);
    const int64_t rows = n_tok * n_heads;
    // every stage's checks before the first launch: after an error nothing is enqueued.  (The sort has
    // none that the sizes and the workspace above leave open.)
    const char* name = "ethos_layer_forward";
    int rc = 0;
    if (n_experts > INT32_MAX || (int64_t)n_sub_keys * n_sub_keys > n_experts)
        return fail(ETHOS_ESIZE, "%s: %d sub-keys give ids past the %lld experts", name, n_sub_keys, (long long)n_experts);
    if (wq_prepared && (rc = query_prepared_checks(name, wq_prepared, wq_prepared_bytes, n_tok, d_model, n_heads, d_query, dtype)))
        return rc;
    if ((rc = query_proj_checks(name, x, wq, wq_prepared, bq, bn_alpha, bn_beta, n_tok, d_model, n_heads, d_query, dtype, w + l.qws,
                                l.qws_bytes, q)))
        return rc;
    if ((rc = route_checks(name, rows, d_query, n_sub_keys, top_k, k_cand, dtype))) return rc;
    if (keys_prepared && (rc = route_prepared_checks(name, keys_prepared, keys_prepared_bytes, d_query, n_sub_keys, dtype))) return rc;
    if ((rc = route_pointer_checks(name, q, sub_keys_1, sub_keys_2, gates, ids))) return rc;
    if ((rc = expert_forward_checks(name, x, latents, n_experts, w1, w2, wut, xp, uniq, seg_off, n_unique, l.max_u, perm, sorted_slot,
                                    pair_slot, gates, n_tok, n_heads, top_k, d_latent, d_hidden, d_model, dtype, order, w + l.ews,
                                    l.ews_bytes, w + l.h, out)))
        return rc;
    rc = wq_prepared ? ethos_query_proj_prepared(x, wq, wq_prepared, wq_prepared_bytes, bq, bn_alpha, bn_beta, n_tok, d_model,
                                                 n_heads, d_query, dtype, w + l.qws, l.qws_bytes, q, stream)
                     : ethos_query_proj(x, wq, bq, bn_alpha, bn_beta, n_tok, d_model, n_heads, d_query, dtype, w + l.qws,
                                        l.qws_bytes, q, stream);
    if (rc) return rc;
    rc = keys_prepared ? ethos_route_topk_prepared(q, sub_keys_1, sub_keys_2, key_norms, keys_prepared, keys_prepared_bytes, rows,
                                                   d_query, n_sub_keys, top_k, k_cand, dtype, gates, ids, stream)
                       : ethos_route_topk(q, sub_keys_1, sub_keys_2, key_norms, rows, d_query, n_sub_keys, top_k, k_cand, dtype,
                                          gates, ids, stream);
    if (rc) return rc;
    if (dtype == ETHOS_BF16 && wut && l.n_pairs <= ETHOS_SMALL_SORT_PAIRS) {  // with the token projection in the sort's launch
        xp = w + l.xp;
        rc = ethos_sort_segment_token_proj(ids, l.n_pairs, n_experts, w + l.shared, l.sort_bytes, perm, uniq, seg_off, pair_slot,
                                           sorted_slot, n_unique, x, w2, wut, n_tok, d_model, d_hidden, dtype, xp, stream);
    } else {
        rc = ethos_sort_segment(ids, l.n_pairs, n_experts, w + l.shared, l.sort_bytes, perm, uniq, seg_off, pair_slot, sorted_slot,
                                n_unique, stream);
    }
    if (rc) return rc;
    return ethos_expert_forward(x, latents, n_experts, w1, w2, wut, xp, uniq, seg_off, n_unique, l.max_u, perm, sorted_slot,
                                pair_slot, gates, n_tok, n_heads, top_k, d_latent, d_hidden, d_model, dtype, order, w + l.ews,
                                l.ews_bytes, w + l.h, out, stream);
}

}  // extern "C"
