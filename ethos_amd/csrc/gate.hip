// Query BatchNorm with batch statistics, and the backward of the routing gates
// (model.py:200-202, 215-234: g = softmax(q1 . K1[i1] + q2 . K2[i2]) over a row's chosen
// experts, with q the per-head BatchNorm of x Wq^T + b, all in float32).
//
// Columns are the C = heads * d_query query channels, rows the tokens (statistics) or the
// (token, head) pairs (gates).  Sums over tokens are float64, in a fixed order: 256-column
// stripes of at most kMaxChunks row chunks each, then the chunks.
//
// 4,096 tokens, 8 heads, d_query 256, bf16: as float32 torch operations differentiated by
// autograd (dense sub-scores, a pass of zeros and a scatter per table, BatchNorm backward
// 178 us) the gates' forward and backward took 2.1 ms, here the backward takes 0.47 ms (queries
// 51 us, rows 82, sub-keys 108, statistics and their backward 48, d Wq 80, dx 97) and the forward
// a copy.  Training-mode queries: one batch_norm call per head 0.59 ms; here the statistics of
// float32 layers 15 us (bf16 layers take torch's, 0.12 ms) and the rest 15 us.
#include "ethos_common.hpp"
#include "ethos_gemm.hpp"
#include "ethos_launch.hpp"

namespace ethos {
namespace {

constexpr int kMaxChunks = 128;

// Per-head parameter tensors [d_query] (the modules own one tensor per head).
struct HeadPtrs {
    const void* gamma[kMaxBnHeads];
    const void* beta[kMaxBnHeads];
    void* mean[kMaxBnHeads];
    void* var[kMaxBnHeads];
    const float* batch_mean[kMaxBnHeads];  // the batch's statistics when the caller has them
    const float* batch_var[kMaxBnHeads];
};

// Four consecutive values as float32.
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load4(const uint16_t* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
}
__device__ __forceinline__ void store4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ __forceinline__ void store4(uint16_t* p, float4 v) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
}

// Column sums of a chunk of rows: of v and v^2, or (GRAD) of g and g * xhat with
// xhat = (v - mean) * invstd.  A lane takes four columns, the four waves every fourth row.
template <typename T, bool GRAD>
__global__ __launch_bounds__(256) void col_sums_kernel(const T* __restrict__ v, const float* __restrict__ g,
                                                       const float* __restrict__ mean, const float* __restrict__ invstd,
                                                       int64_t n, int cols, int64_t per, double2* __restrict__ part) {
    __shared__ double2 lds[3][64][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c0 = blockIdx.x * 256 + lane * 4;
    const int c = c0 < cols ? c0 : cols - 4;
    const int64_t r0 = blockIdx.y * per, r1 = r0 + per < n ? r0 + per : n;
    double s[4] = {0, 0, 0, 0}, t[4] = {0, 0, 0, 0};
    float4 mu = make_float4(0, 0, 0, 0), is = mu;
    if (GRAD) {
        mu = load4(mean + c);
        is = load4(invstd + c);
    }
    constexpr int U = 4;
    for (int64_t r = r0 + wave; r < r1; r += 4 * U) {
        float4 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t rr = r + 4 * u < r1 ? r + 4 * u : r;
            a[u] = load4(v + rr * cols + c);
            if (GRAD) b[u] = load4(g + rr * cols + c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (r + 4 * u >= r1) break;
            const float av[4] = {a[u].x, a[u].y, a[u].z, a[u].w};
            if (GRAD) {
                const float bv[4] = {b[u].x, b[u].y, b[u].z, b[u].w};
                const float m4[4] = {mu.x, mu.y, mu.z, mu.w}, i4[4] = {is.x, is.y, is.z, is.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s[j] += (double)bv[j];
                    t[j] = fma((double)bv[j], (double)((av[j] - m4[j]) * i4[j]), t[j]);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s[j] += (double)av[j];
                    t[j] = fma((double)av[j], (double)av[j], t[j]);
                }
            }
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) lds[wave - 1][lane][j] = make_double2(s[j], t[j]);
    }
    __syncthreads();
    if (wave == 0 && c0 < cols) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            for (int w = 0; w < 3; ++w) {
                s[j] += lds[w][lane][j].x;
                t[j] += lds[w][lane][j].y;
            }
            part[(int64_t)blockIdx.y * cols + c0 + j] = make_double2(s[j], t[j]);
        }
    }
}

// Sum of a column's chunks, 16 lanes a column; the total in every lane of the 16.
__device__ __forceinline__ double2 sum_chunks(const double2* __restrict__ part, int chunks, int cols, int col) {
    __shared__ double2 lds[16][17];
    const int l = threadIdx.x & 15, q = threadIdx.x >> 4;
    double2 v[kMaxChunks / 16];
#pragma unroll
    for (int i = 0; i < kMaxChunks / 16; ++i) {
        const int k = l + 16 * i;
        v[i] = part[(int64_t)(k < chunks ? k : chunks - 1) * cols + col];
    }
    double2 s = make_double2(0, 0);
#pragma unroll
    for (int i = 0; i < kMaxChunks / 16; ++i) {
        if (l + 16 * i < chunks) {
            s.x += v[i].x;
            s.y += v[i].y;
        }
    }
    lds[q][l] = s;
    __syncthreads();
    s = make_double2(0, 0);
    for (int i = 0; i < 16; ++i) {
        s.x += lds[q][i].x;
        s.y += lds[q][i].y;
    }
    return s;
}

// Per column: mean, 1 / sqrt(var + eps), gamma and beta as float32, from the batch (chunk sums;
// with `update`, the running statistics too: (1 - momentum) running + momentum batch, the
// variance unbiased), from the batch's statistics of the caller (`given`), or from the running
// statistics.  16 columns per workgroup of 256.
template <typename T>
__global__ __launch_bounds__(256) void bn_stats_kernel(const double2* __restrict__ part, int chunks, int64_t n, int cols, int dq,
                                                       HeadPtrs hp, int given, int update, double momentum, double eps,
                                                       float* __restrict__ out) {
    const int col0 = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int col = col0 < cols ? col0 : cols - 1;
    const int h = col / dq, e = col % dq;
    double mu, var;
    if (given) {
        mu = hp.batch_mean[h][e];
        var = hp.batch_var[h][e];
    } else if (part) {
        const double2 s = sum_chunks(part, chunks, cols, col);
        mu = s.x / (double)n;
        var = s.y / (double)n - mu * mu;
        var = var > 0.0 || !(var == var) ? var : 0.0;
    } else {
        mu = Elem<T>::to_f64(((const T*)hp.mean[h])[e]);
        var = Elem<T>::to_f64(((const T*)hp.var[h])[e]);
    }
    if ((threadIdx.x & 15) != 0 || col0 >= cols) return;
    out[col] = (float)mu;
    out[cols + col] = given ? rsqrtf((float)var + (float)eps) : (float)(1.0 / sqrt(var + eps));
    out[2 * cols + col] = Elem<T>::to_f32(((const T*)hp.gamma[h])[e]);
    out[3 * cols + col] = Elem<T>::to_f32(((const T*)hp.beta[h])[e]);
    if (update) {
        T *rm = (T*)hp.mean[h] + e, *rv = (T*)hp.var[h] + e;
        const double unbiased = var * ((double)n / (double)(n - 1));
        *rm = Elem<T>::from_f32((float)(momentum * mu + (1.0 - momentum) * Elem<T>::to_f64(*rm)));
        *rv = Elem<T>::from_f32((float)(momentum * unbiased + (1.0 - momentum) * Elem<T>::to_f64(*rv)));
    }
}

// q = RN_T((v - mean) gamma invstd + beta).
template <typename T>
__global__ __launch_bounds__(256) void bn_apply_kernel(const T* __restrict__ v, const float* __restrict__ st, int64_t n, int cols,
                                                       T* __restrict__ q) {
    const int64_t total = n * (cols / 4);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int c = (int)(i % (cols / 4)) * 4;
        const float4 a = load4(v + i * 4), mu = load4(st + c), is = load4(st + cols + c), ga = load4(st + 2 * cols + c),
                     be = load4(st + 3 * cols + c);
        store4(q + i * 4, make_float4(__builtin_fmaf((a.x - mu.x) * ga.x, is.x, be.x), __builtin_fmaf((a.y - mu.y) * ga.y, is.y, be.y),
                                      __builtin_fmaf((a.z - mu.z) * ga.z, is.z, be.z), __builtin_fmaf((a.w - mu.w) * ga.w, is.w, be.w)));
    }
}

// V consecutive values as float32.
template <typename T, int V>
__device__ __forceinline__ void load_v(const T* p, float* v) {
    if constexpr (V >= 4) {
#pragma unroll
        for (int i = 0; i < V; i += 4) {
            const float4 f = load4(p + i);
            v[i] = f.x, v[i + 1] = f.y, v[i + 2] = f.z, v[i + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] = Elem<T>::to_f32(p[i]);
    }
}

// A wave's own LDS accesses complete in order; this keeps the compiler from reordering them.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One wave per (token, head) row: lanes 0..31 hold the first query half (V values each), lanes
// 32..63 the second, so that a pair's two sub-key rows are one load and its score one sum over
// the wave.  Lane p < k keeps pair p's score: softmax, then ds = g (dg - sum g dg).  Writes the
// row's normalised query, its gradient sum_p ds_p K[i_p], and ds spread over the 2 K sub-keys
// (the pairs that share a sub-key added up in pair order), the left operand of the sub-keys'
// gradient.  Bound by its L2 reads (the sub-key rows, twice) and the 4 (2 dq + 2 K) bytes a
// row that it writes.
template <typename T, int V>
__global__ __launch_bounds__(256) void gate_rows_kernel(const float* __restrict__ qf, const float* __restrict__ st,
                                                        const T* __restrict__ k1, const T* __restrict__ k2,
                                                        const int32_t* __restrict__ ids, const float* __restrict__ dg, int64_t rows,
                                                        int H, int dq, int K, int pitch, int k, float* __restrict__ qn,
                                                        float* __restrict__ dqn, float* __restrict__ ds) {
    extern __shared__ float lds_ds[];
    constexpr int G = 8;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* mine = lds_ds + wave * 2 * pitch;
    const int half = dq / 2, cols = H * dq;
    const bool second = lane >= 32;
    const int e = (lane & 31) * V;
    const bool in = e < half;
    const int ee = in ? e : 0;
    const T* table = second ? k2 : k1;
    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < rows; r += (int64_t)gridDim.x * 4) {
        const int h = (int)(r % H);
        const int c = h * dq + (second ? half : 0) + ee;
        const int64_t at = r * dq + (second ? half : 0) + ee;
        float q[V], mu[V], is[V], ga[V], be[V];
        load_v<float, V>(qf + at, q);
        load_v<float, V>(st + c, mu);
        load_v<float, V>(st + cols + c, is);
        load_v<float, V>(st + 2 * cols + c, ga);
        load_v<float, V>(st + 3 * cols + c, be);
        const int my = lane < k ? lane : k - 1;
        const int id = ids[r * k + my];
        const float my_dg = dg[r * k + my];
        const int my1 = id / K, my2 = id - my1 * K;
#pragma unroll
        for (int v = 0; v < V; ++v) q[v] = in ? __builtin_fmaf((q[v] - mu[v]) * is[v], ga[v], be[v]) : 0.0f;
        float score = -INFINITY;
        for (int p0 = 0; p0 < k; p0 += G) {
            float kv[G][V];
#pragma unroll
            for (int u = 0; u < G; ++u) {
                const int p = p0 + u < k ? p0 + u : k - 1;
                const int row = second ? __builtin_amdgcn_readlane(my2, p) : __builtin_amdgcn_readlane(my1, p);
                load_v<T, V>(table + (int64_t)row * half + ee, kv[u]);
            }
#pragma unroll
            for (int u = 0; u < G; ++u) {
                float d = 0.0f;
#pragma unroll
                for (int v = 0; v < V; ++v) d = __builtin_fmaf(q[v], kv[u][v], d);
                const float s = wave_sum(d);
                score = lane == p0 + u && p0 + u < k ? s : score;
            }
        }
        float top = score;
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) top = fmaxf(top, __shfl_xor(top, m, 64));
        const float ex = lane < k ? expf(score - top) : 0.0f;
        const float g = ex / wave_sum(ex);
        const float dot = wave_sum(lane < k ? g * my_dg : 0.0f);
        const float my_ds = lane < k ? g * (my_dg - dot) : 0.0f;

        // the row of ds over the sub-keys
        wave_lds_fence();
        for (int i = lane * 4; i < 2 * pitch; i += 256) *reinterpret_cast<float4*>(mine + i) = make_float4(0, 0, 0, 0);
        float s1 = 0.0f, s2 = 0.0f;
        for (int p = 0; p < k; ++p) {
            const float d = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_ds), p));
            s1 += __builtin_amdgcn_readlane(my1, p) == my1 ? d : 0.0f;
            s2 += __builtin_amdgcn_readlane(my2, p) == my2 ? d : 0.0f;
        }
        wave_lds_fence();
        if (lane < k) {
            mine[my1] = s1;
            mine[pitch + my2] = s2;
        }
        wave_lds_fence();
        for (int i = lane * 4; i < 2 * pitch; i += 256)
            *reinterpret_cast<float4*>(ds + r * 2 * pitch + i) = *reinterpret_cast<const float4*>(mine + i);

        float dv[V];
#pragma unroll
        for (int v = 0; v < V; ++v) dv[v] = 0.0f;
        for (int p0 = 0; p0 < k; p0 += G) {
            float kv[G][V];
#pragma unroll
            for (int u = 0; u < G; ++u) {
                const int p = p0 + u < k ? p0 + u : k - 1;
                const int row = second ? __builtin_amdgcn_readlane(my2, p) : __builtin_amdgcn_readlane(my1, p);
                load_v<T, V>(table + (int64_t)row * half + ee, kv[u]);
            }
#pragma unroll
            for (int u = 0; u < G; ++u) {
                if (p0 + u >= k) break;
                const float d = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_ds), p0 + u));
#pragma unroll
                for (int v = 0; v < V; ++v) dv[v] = __builtin_fmaf(d, kv[u][v], dv[v]);
            }
        }
        if (in) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                qn[at + v] = q[v];
                dqn[at + v] = dv[v];
            }
        }
    }
}

// Per column, from the chunk sums S = sum dqn and X = sum dqn xhat: d beta = S, d gamma = X, the
// terms S / n and X / n that batch statistics take off each row's gradient (zero otherwise), and
// d bias: gamma invstd S with running statistics, zero (0 S, so that a NaN shows) with the
// batch's, which take the bias away.
template <typename T>
__global__ __launch_bounds__(256) void bn_grad_sums_kernel(const double2* __restrict__ part, int chunks, int64_t n, int cols,
                                                           int batch, const float* __restrict__ st, float* __restrict__ sub,
                                                           T* __restrict__ dgamma, T* __restrict__ dbeta, T* __restrict__ dbias) {
    const int col0 = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int col = col0 < cols ? col0 : cols - 1;
    const double2 s = sum_chunks(part, chunks, cols, col);
    if ((threadIdx.x & 15) != 0 || col0 >= cols) return;
    dbeta[col] = Elem<T>::from_f32((float)s.x);
    dgamma[col] = Elem<T>::from_f32((float)s.y);
    dbias[col] = Elem<T>::from_f32(batch ? 0.0f * (float)s.x : (float)(s.x * (double)st[2 * cols + col] * (double)st[cols + col]));
    sub[col] = batch ? (float)(s.x / (double)n) : 0.0f;
    sub[cols + col] = batch ? (float)(s.y / (double)n) : 0.0f;
}

// The gradient before BatchNorm, in place: gamma invstd (dqn - S / n - xhat X / n).
__global__ __launch_bounds__(256) void bn_grad_apply_kernel(const float* __restrict__ qf, const float* __restrict__ st,
                                                            const float* __restrict__ sub, int64_t n, int cols,
                                                            float* __restrict__ dq) {
    const int64_t total = n * (cols / 4);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int c = (int)(i % (cols / 4)) * 4;
        const float4 a = load4(qf + i * 4), d = load4(dq + i * 4), mu = load4(st + c), is = load4(st + cols + c),
                     ga = load4(st + 2 * cols + c), s = load4(sub + c), x = load4(sub + cols + c);
        store4(dq + i * 4, make_float4(ga.x * is.x * (d.x - s.x - (a.x - mu.x) * is.x * x.x),
                                       ga.y * is.y * (d.y - s.y - (a.y - mu.y) * is.y * x.y),
                                       ga.z * is.z * (d.z - s.z - (a.z - mu.z) * is.z * x.z),
                                       ga.w * is.w * (d.w - s.w - (a.w - mu.w) * is.w * x.w)));
    }
}

// alpha = fp32(gamma / sqrt(var + eps)), beta' = fp32(beta - mean alpha), each in float64 and
// rounded once (float64 sqrt and division are correctly rounded on the device too).
template <typename T>
__global__ __launch_bounds__(256) void bn_coefficients_kernel(HeadPtrs hp, int cols, int dq, double eps, float* __restrict__ alpha,
                                                              float* __restrict__ beta) {
    const int col = blockIdx.x * 256 + threadIdx.x;
    if (col >= cols) return;
    const int h = col / dq, e = col % dq;
    const double w = hp.gamma[h] ? Elem<T>::to_f64(((const T*)hp.gamma[h])[e]) : 1.0;
    const double b = hp.beta[h] ? Elem<T>::to_f64(((const T*)hp.beta[h])[e]) : 0.0;
    const double mu = hp.mean[h] ? Elem<T>::to_f64(((const T*)hp.mean[h])[e]) : 0.0;
    const double var = hp.var[h] ? Elem<T>::to_f64(((const T*)hp.var[h])[e]) : 1.0;
    const float a = (float)(w / sqrt(var + eps));
    alpha[col] = a;
    // the product, then the difference, each rounded to float64
    const double ma = __dmul_rn(mu, (double)a);
    beta[col] = (float)__dadd_rn(b, -ma);
}

struct Chunks {
    int count;
    int64_t per;
};
Chunks row_chunks(int64_t n) {
    int64_t per = (n + kMaxChunks - 1) / kMaxChunks;
    per = per < 32 ? 32 : per;
    return {(int)((n + per - 1) / per), per};
}

size_t pad256(size_t n) { return (n + 255) & ~(size_t)255; }
unsigned grid1(int64_t items, int num_cus) {
    int64_t b = (items + 255) / 256;
    const int64_t cap = (int64_t)num_cus * 16;
    return (unsigned)(b < cap ? (b < 1 ? 1 : b) : cap);
}

HeadPtrs head_ptrs(const void* const* gamma, const void* const* beta, void* const* mean, void* const* var, int H,
                   const float* const* batch_mean = nullptr, const float* const* batch_var = nullptr) {
    HeadPtrs p{};
    for (int h = 0; h < H; ++h) {
        p.gamma[h] = gamma ? gamma[h] : nullptr;
        p.beta[h] = beta ? beta[h] : nullptr;
        p.mean[h] = mean ? mean[h] : nullptr;
        p.var[h] = var ? var[h] : nullptr;
        p.batch_mean[h] = batch_mean ? batch_mean[h] : nullptr;
        p.batch_var[h] = batch_var ? batch_var[h] : nullptr;
    }
    return p;
}

template <typename T>
int query_bn_t(const T* v, int64_t n, int H, int dq, const HeadPtrs& hp, int given, int update, double momentum, double eps, void* ws, T* q,
               int num_cus, hipStream_t stream) {
    const int cols = H * dq;
    const Chunks ch = row_chunks(n);
    double2* part = (double2*)ws;
    float* st = (float*)((unsigned char*)ws + pad256((size_t)ch.count * cols * sizeof(double2)));
    if (!given)
        hipLaunchKernelGGL((col_sums_kernel<T, false>), dim3((cols + 255) / 256, ch.count), dim3(256), 0, stream, v,
                       (const float*)nullptr, (const float*)nullptr, (const float*)nullptr, n, cols, ch.per, part);
    hipLaunchKernelGGL((bn_stats_kernel<T>), dim3((cols + 15) / 16), dim3(256), 0, stream, (const double2*)part, ch.count, n, cols,
                       dq, hp, given, update, momentum, eps, st);
    hipLaunchKernelGGL((bn_apply_kernel<T>), dim3(grid1(n * (cols / 4), num_cus)), dim3(256), 0, stream, v, (const float*)st, n,
                       cols, q);
    return (int)hipGetLastError();
}

struct GateLayout {
    size_t qf, qn, dqn, ds, part, st, sub, gpart, total;
    int pitch, split_w, split_k;
};
GateLayout gate_layout(int64_t n, int H, int k, int d, int dq, int K, int num_cus) {
    GateLayout l{};
    const int cols = H * dq;
    const size_t rows = pad256((size_t)n * cols * sizeof(float));
    l.pitch = (K + 3) / 4 * 4;
    l.split_w = gemm_split(cols, d, n, num_cus);
    l.split_k = gemm_split(K, dq / 2, n * H, num_cus);
    l.qf = 0;
    l.qn = rows;
    l.dqn = 2 * rows;
    l.ds = 3 * rows;
    l.part = l.ds + pad256((size_t)n * H * 2 * l.pitch * sizeof(float));
    l.st = l.part + pad256((size_t)row_chunks(n).count * cols * sizeof(double2));
    l.sub = l.st + pad256((size_t)4 * cols * sizeof(float));
    l.gpart = l.sub + pad256((size_t)2 * cols * sizeof(float));
    const size_t pw = l.split_w > 1 ? (size_t)l.split_w * cols * d : 0, pk = l.split_k > 1 ? (size_t)l.split_k * K * (dq / 2) : 0;
    l.total = l.gpart + pad256((pw > pk ? pw : pk) * sizeof(float));
    return l;
}

template <typename T, int V>
void launch_rows(const float* qf, const float* st, const T* k1, const T* k2, const int32_t* ids, const float* dg, int64_t rows, int H,
                 int dq, int K, int pitch, int k, float* qn, float* dqn, float* ds, int num_cus, hipStream_t stream) {
    int64_t b = (rows + 3) / 4;
    const int64_t cap = (int64_t)num_cus * 16;
    b = b < cap ? b : cap;
    hipLaunchKernelGGL((gate_rows_kernel<T, V>), dim3((unsigned)b), dim3(256), 4 * 2 * pitch * sizeof(float), stream, qf, st, k1, k2,
                       ids, dg, rows, H, dq, K, pitch, k, qn, dqn, ds);
}

template <typename T>
int gate_grads_t(const T* x, const int32_t* ids, const float* dg, const T* wq, const T* bq, const T* k1, const T* k2,
                 const HeadPtrs& hp, int batch, double eps, int64_t n, int d, int H, int dq, int K, int k, void* ws, T* dx, T* dw,
                 T* db, T* dgamma, T* dbeta, T* dk1, T* dk2, int num_cus, hipStream_t stream) {
    constexpr bool bf = sizeof(T) == 2;
    const GateLayout l = gate_layout(n, H, k, d, dq, K, num_cus);
    const int cols = H * dq, half = dq / 2;
    unsigned char* w = (unsigned char*)ws;
    float *qf = (float*)(w + l.qf), *qn = (float*)(w + l.qn), *dqn = (float*)(w + l.dqn), *ds = (float*)(w + l.ds);
    double2* part = (double2*)(w + l.part);
    float *st = (float*)(w + l.st), *sub = (float*)(w + l.sub), *gpart = (float*)(w + l.gpart);
    int rc;

    Gemm g;  // queries before BatchNorm
    g.a = x, g.lda = d, g.b = wq, g.ldb = d, g.c = qf, g.ldc = cols, g.bias = bq;
    g.m = n, g.n = cols, g.k = d;
    if ((rc = launch_gemm(bf ? kGemmBK_BK : kGemmFK_FK, g, num_cus, stream))) return rc;

    const Chunks ch = row_chunks(n);
    const dim3 sums((cols + 255) / 256, ch.count), per_col((cols + 15) / 16);
    if (batch)
        hipLaunchKernelGGL((col_sums_kernel<float, false>), sums, dim3(256), 0, stream, (const float*)qf, (const float*)nullptr,
                           (const float*)nullptr, (const float*)nullptr, n, cols, ch.per, part);
    hipLaunchKernelGGL((bn_stats_kernel<T>), per_col, dim3(256), 0, stream, batch ? (const double2*)part : nullptr, ch.count, n, cols,
                       dq, hp, 0, 0, 0.0, eps, st);
    const int v = (half + 31) / 32;
#define ETHOS_GATE_ROWS(VV)                                                                                                     \
    launch_rows<T, VV>(qf, st, k1, k2, ids, dg, n * H, H, dq, K, l.pitch, k, qn, dqn, ds, num_cus, stream)
    if (v <= 1) ETHOS_GATE_ROWS(1);
    else if (v <= 2) ETHOS_GATE_ROWS(2);
    else if (v <= 4) ETHOS_GATE_ROWS(4);
    else ETHOS_GATE_ROWS(8);
#undef ETHOS_GATE_ROWS

    for (int i = 0; i < 2; ++i) {  // d K_i = ds_i^T q_i over the rows
        g = Gemm{};
        g.a = ds + i * l.pitch, g.lda = 2 * l.pitch, g.b = qn + i * half, g.ldb = dq, g.c = i ? dk2 : dk1, g.ldc = half;
        g.m = K, g.n = half, g.k = n * H, g.out_bf16 = bf, g.split = l.split_k, g.part = gpart;
        if ((rc = launch_gemm(kGemmFR_FR, g, num_cus, stream))) return rc;
    }

    hipLaunchKernelGGL((col_sums_kernel<float, true>), sums, dim3(256), 0, stream, (const float*)qf, (const float*)dqn,
                       (const float*)st, (const float*)(st + cols), n, cols, ch.per, part);
    hipLaunchKernelGGL((bn_grad_sums_kernel<T>), per_col, dim3(256), 0, stream, (const double2*)part, ch.count, n, cols, batch,
                       (const float*)st, sub, dgamma, dbeta, db);
    hipLaunchKernelGGL(bn_grad_apply_kernel, dim3(grid1(n * (cols / 4), num_cus)), dim3(256), 0, stream, (const float*)qf,
                       (const float*)st, (const float*)sub, n, cols, dqn);

    g = Gemm{};  // d Wq = dq^T x
    g.a = dqn, g.lda = cols, g.b = x, g.ldb = d, g.c = dw, g.ldc = d;
    g.m = cols, g.n = d, g.k = n, g.out_bf16 = bf, g.split = l.split_w, g.part = gpart;
    if (dw && (rc = launch_gemm(bf ? kGemmFR_BR : kGemmFR_FR, g, num_cus, stream))) return rc;
    if (!dx) return (int)hipGetLastError();

    g = Gemm{};  // dx = dq Wq
    g.a = dqn, g.lda = cols, g.b = wq, g.ldb = d, g.c = dx, g.ldc = d;
    g.m = n, g.n = d, g.k = cols, g.out_bf16 = bf;
    return launch_gemm(bf ? kGemmFK_BR : kGemmFK_FR, g, num_cus, stream);
}

}  // namespace

size_t query_bn_workspace_bytes(int64_t n, int H, int dq) {
    const int cols = H * dq;
    return pad256((size_t)row_chunks(n).count * cols * sizeof(double2)) + pad256((size_t)4 * cols * sizeof(float));
}

int launch_query_bn(const void* v, int64_t n, int H, int dq, int dtype, const void* const* gamma, const void* const* beta,
                    void* const* mean, void* const* var, const float* const* batch_mean, const float* const* batch_var,
                    double momentum, double eps, void* ws, void* q, int num_cus, hipStream_t stream) {
    const HeadPtrs hp = head_ptrs(gamma, beta, mean, var, H, batch_mean, batch_var);
    const int given = batch_mean != nullptr;
    const int update = mean != nullptr;
    if (dtype == kBF16)
        return query_bn_t((const uint16_t*)v, n, H, dq, hp, given, update, momentum, eps, ws, (uint16_t*)q, num_cus, stream);
    return query_bn_t((const float*)v, n, H, dq, hp, given, update, momentum, eps, ws, (float*)q, num_cus, stream);
}

int launch_bn_coefficients(int H, int dq, int dtype, const void* const* gamma, const void* const* beta, void* const* mean,
                           void* const* var, double eps, float* alpha, float* shift, hipStream_t stream) {
    const HeadPtrs hp = head_ptrs(gamma, beta, mean, var, H);
    const int cols = H * dq;
    if (dtype == kBF16)
        hipLaunchKernelGGL((bn_coefficients_kernel<uint16_t>), dim3((cols + 255) / 256), dim3(256), 0, stream, hp, cols, dq, eps,
                           alpha, shift);
    else
        hipLaunchKernelGGL((bn_coefficients_kernel<float>), dim3((cols + 255) / 256), dim3(256), 0, stream, hp, cols, dq, eps,
                           alpha, shift);
    return (int)hipGetLastError();
}

// A lane's values of the query half are whole (V = 1, 2, 4 or 8 of half / V lanes).
bool gate_grads_supported(int H, int dq, int K, int k) {
    const int half = dq / 2, v = (half + 31) / 32, V = v <= 1 ? 1 : v <= 2 ? 2 : v <= 4 ? 4 : 8;
    return H <= kMaxBnHeads && dq % 8 == 0 && half <= 256 && half % V == 0 && K <= 1024 && k <= 64;
}

size_t gate_grads_workspace_bytes(int64_t n, int H, int k, int d, int dq, int K, int num_cus) {
    return gate_layout(n, H, k, d, dq, K, num_cus).total;
}

int launch_gate_grads(const void* x, const int32_t* ids, const float* dg, const void* wq, const void* bq, const void* k1,
                      const void* k2, const void* const* gamma, const void* const* beta, void* const* mean, void* const* var,
                      double eps, int64_t n, int d, int H, int dq, int K, int k, int dtype, void* ws, void* dx, void* dw, void* db,
                      void* dgamma, void* dbeta, void* dk1, void* dk2, int num_cus, hipStream_t stream) {
    const HeadPtrs hp = head_ptrs(gamma, beta, mean, var, H);
    const int batch = mean == nullptr;
    if (dtype == kBF16) {
        using T = uint16_t;
        return gate_grads_t((const T*)x, ids, dg, (const T*)wq, (const T*)bq, (const T*)k1, (const T*)k2, hp, batch, eps, n, d, H, dq,
                            K, k, ws, (T*)dx, (T*)dw, (T*)db, (T*)dgamma, (T*)dbeta, (T*)dk1, (T*)dk2, num_cus, stream);
    }
    using T = float;
    return gate_grads_t((const T*)x, ids, dg, (const T*)wq, (const T*)bq, (const T*)k1, (const T*)k2, hp, batch, eps, n, d, H, dq, K,
                        k, ws, (T*)dx, (T*)dw, (T*)db, (T*)dgamma, (T*)dbeta, (T*)dk1, (T*)dk2, num_cus, stream);
}

}  // namespace ethos
