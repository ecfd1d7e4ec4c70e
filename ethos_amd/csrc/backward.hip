// Backward of the expert stages: the derivative of the reference layer's per-pair
// expression (model.py:312-341, differentiated by autograd there; the reference's Triton
// layer, kernels.py:145-221, has no backward).
//
// With A = W2[:d] and B = W2[d:] (net.2.weight halves), pair p of token t(p) using unique
// expert s(p), c_p = h_s . xp_t, a_p = gelu(c_p) g_p and dY_t = dy_t / H, the per-pair part
// of the backward is, given xp = x A and dYB = dY B (both float32 [n_tok, d_hidden]):
//
//   da_p  = dYB_t . h_s                 (= dY_t . v_s with v_s = h_s B^T)
//   dg_p  = gelu(c_p) da_p
//   dc_p  = g_p gelu'(c_p) da_p
//   hacc_t = sum_p a_p h_s,   dxp_t = sum_p dc_p h_s                       (token sums)
//   dh_s  += a_p dYB_t + dc_p xp_t                                          (expert sums)
//
// Three kernels, all deterministic (every sum has a fixed order, no atomics):
//  1. expert_bwd_pairs_kernel: one wave per token walks its H k pairs (bwd_unroll hidden
//     rows in flight), keeps xp_t, dYB_t and the token sums in registers, and stores each
//     pair's scalars (a_p, dc_p);
//  2. expert_bwd_sums_kernel: the expert sums over the sorted pairs (ethos_sort_segment's
//     permutation, each expert's pairs consecutive and in pair order), a quarter wave per
//     block of kBwdBlock sorted positions and 64 columns, summing each segment's terms in sorted order: a
//     segment that lies in one block is written to dh; a segment crossing blocks leaves
//     its part in its first block (tail) and in each later block (head) as partial rows;
//  3. expert_bwd_join_kernel: each crossing segment's dh = its first block's tail part plus
//     the later blocks' head parts, in block order.
// launch_expert_grads runs the whole node: xp and dYB first, then these kernels, then the
// weight, input and latent gradients as float32 matrix products (gemm.hip).
#include <algorithm>

#include "ethos_common.hpp"
#include "ethos_gelu.hpp"
#include "ethos_gemm.hpp"
#include "ethos_launch.hpp"
#include "ethos_rows.hpp"

namespace ethos {

// Hidden rows in flight per wave: fewer for rows of many registers.
constexpr int bwd_unroll(int ch) { return ch <= 2 ? 8 : ch == 4 ? 4 : 2; }

constexpr int kBwdBlock = 64;  // sorted positions per block of the expert-sum pass

template <typename T, int CH>
__global__ __launch_bounds__(256) void expert_bwd_pairs_kernel(const T* __restrict__ hid, const float* __restrict__ xp,
                                                               const float* __restrict__ dyb,
                                                               const int32_t* __restrict__ pair_slot,
                                                               const T* __restrict__ gates, int64_t n_tok, int hk,
                                                               int dh, float* __restrict__ dg,
                                                               float* __restrict__ hacc, float* __restrict__ dxp,
                                                               float2* __restrict__ ac) {
    constexpr int N = Vec16<T>::kN;
    constexpr int kBwdUnroll = bwd_unroll(CH);
    typedef typename Vec16<T>::raw Raw;
    const int lane = threadIdx.x & 63;
    const int64_t wave_id = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n_waves = (int64_t)gridDim.x * 4;
    for (int64_t t = wave_id; t < n_tok; t += n_waves) {
        float xr[CH * N], yr[CH * N], ha[CH * N], dx[CH * N];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int e = c * 64 * N + lane * N;
#pragma unroll
            for (int v = 0; v < N; ++v) {
                const bool in = e + v < dh;
                xr[c * N + v] = in ? xp[t * dh + e + v] : 0.0f;
                yr[c * N + v] = in ? dyb[t * dh + e + v] : 0.0f;
                ha[c * N + v] = 0.0f;
                dx[c * N + v] = 0.0f;
            }
        }
        const int64_t pbase = t * hk;
        for (int j0 = 0; j0 < hk; j0 += kBwdUnroll) {
            Raw hr[kBwdUnroll][CH];
            int sq[kBwdUnroll];
            // slots first, then every row with no branch between the loads (past the last pair
            // the last pair's row again, unused)
#pragma unroll
            for (int q = 0; q < kBwdUnroll; ++q) sq[q] = pair_slot[pbase + (j0 + q < hk ? j0 + q : hk - 1)];
#pragma unroll
            for (int q = 0; q < kBwdUnroll; ++q) load_raw_buf<T, CH>(hid + (int64_t)sq[q] * dh, dh, lane, hr[q]);
            // lane q's pair: its gate, then its two dot products, so that the GELU and its derivative
            // are evaluated once for the group (for every pair by every lane they took 100 us at
            // 524,288 pairs)
            const int mine = j0 + lane < hk ? j0 + lane : hk - 1;
            const float g = Elem<T>::to_f32(gates[pbase + mine]);
            float my_c = 0.0f, my_d = 0.0f;
#pragma unroll
            for (int q = 0; q < kBwdUnroll; ++q) {
                float hf[CH * N];
                float cp = 0.0f, dp = 0.0f;
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    Vec16<T>::unpack(hr[q][c], hf + c * N);
#pragma unroll
                    for (int v = 0; v < N; ++v) {
                        cp = __builtin_fmaf(hf[c * N + v], xr[c * N + v], cp);
                        dp = __builtin_fmaf(hf[c * N + v], yr[c * N + v], dp);
                    }
                }
                const float cdot = wave_sum(cp), da = wave_sum(dp);
                my_c = lane == q ? cdot : my_c;
                my_d = lane == q ? da : my_d;
            }
            const float act = gelu_erf(my_c);
            const float my_a = act * g;
            const float my_dc = g * gelu_erf_grad(my_c) * my_d;
            if (lane < kBwdUnroll && j0 + lane < hk) {
                dg[pbase + mine] = act * my_d;
                ac[pbase + mine] = make_float2(my_a, my_dc);
            }
#pragma unroll
            for (int q = 0; q < kBwdUnroll; ++q) {
                if (j0 + q >= hk) continue;
                const float a = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_a), q));
                const float dc = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_dc), q));
                float hf[CH * N];
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    Vec16<T>::unpack(hr[q][c], hf + c * N);
#pragma unroll
                    for (int v = 0; v < N; ++v) {
                        ha[c * N + v] = __builtin_fmaf(a, hf[c * N + v], ha[c * N + v]);
                        dx[c * N + v] = __builtin_fmaf(dc, hf[c * N + v], dx[c * N + v]);
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int e = c * 64 * N + lane * N;
            if (e < dh) {
#pragma unroll
                for (int v = 0; v < N; ++v) {
                    hacc[t * dh + e + v] = ha[c * N + v];
                    dxp[t * dh + e + v] = dx[c * N + v];
                }
            }
        }
    }
}

// Expert sums.  A quarter wave (16 lanes, 4 columns each) takes one block of kBwdBlock sorted
// positions for one slice of 64 columns, one position at a time in sorted order; 16 positions'
// pairs, tokens and scalars are loaded a lane each and broadcast over the quarter (DPP), and
// kSumUnroll positions' row pieces are requested together.  A segment's sum is stored when the
// walk leaves it: to dh when the segment lies in the block, else as the block's head part (the
// segment that began before the block) or tail part (the segment that begins in the block and
// continues past it).
// What bounds it is the row gathers, two of 4 d_hidden bytes per pair: 2.1 GB for 524,288 pairs
// at d_hidden 512, out of two tables of 8 MB.  Workgroup b works on slice b % (slices), and runs
// on XCD b % 8, so at 512 columns each XCD's gathers stay in 2 MB of the tables, inside its L2:
// 278 us (one wave per block over all columns, 7.5 TB/s out of the memory-side cache) -> 173 us.
// 16,000 pairs (500 tokens): 113 -> 18 us, a wave's 64 positions no longer one load after another.
constexpr int kSumUnroll = 8;
constexpr int kSumSlice = 64;

// Lane i of each row of 16 to the whole row.
template <int I>
__device__ __forceinline__ int row_bcast(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + I, 0xf, 0xf, false);
}

// Four floats at any float's address (one 16-byte access; callers' xp, dyb and dh need no more
// than their own alignment).
typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 load_any4(const float* p) {
    const f32x4_any_t v = *reinterpret_cast<const f32x4_any_t*>(p);
    return make_float4(v.x, v.y, v.z, v.w);
}

struct SumPos {  // a lane's position
    int t, s, to;   // token, slot, and after this position: 0 go on, 1 store to dh, 2 to head, 3 to tail
    float a, dc;
};

template <int I>
struct SumStep {
    // positions I .. I + kSumUnroll - 1 of the 16
    __device__ __forceinline__ static void run(const SumPos& me, const float* __restrict__ xp, const float* __restrict__ dyb,
                                               int dh, int col, bool in, float4& acc, float* __restrict__ dhs,
                                               float* head, float* tail) {
        float4 x[kSumUnroll], y[kSumUnroll];
        load<0>(me, xp, dyb, dh, col, x, y);
        add<0>(me, dh, col, in, acc, x, y, dhs, head, tail);
    }
    template <int U>
    __device__ __forceinline__ static void load(const SumPos& me, const float* xp, const float* dyb, int dh, int col, float4* x,
                                                float4* y) {
        if constexpr (U < kSumUnroll) {
            const int64_t at = (int64_t)row_bcast<I + U>(me.t) * dh + col;
            y[U] = load_any4(dyb + at);
            x[U] = load_any4(xp + at);
            load<U + 1>(me, xp, dyb, dh, col, x, y);
        }
    }
    template <int U>
    __device__ __forceinline__ static void add(const SumPos& me, int dh, int col, bool in, float4& acc, const float4* x,
                                               const float4* y, float* dhs, float* head, float* tail) {
        if constexpr (U < kSumUnroll) {
            const float a = __int_as_float(row_bcast<I + U>(__float_as_int(me.a)));
            const float dc = __int_as_float(row_bcast<I + U>(__float_as_int(me.dc)));
            const int to = row_bcast<I + U>(me.to), s = row_bcast<I + U>(me.s);
            acc.x = __builtin_fmaf(dc, x[U].x, __builtin_fmaf(a, y[U].x, acc.x));
            acc.y = __builtin_fmaf(dc, x[U].y, __builtin_fmaf(a, y[U].y, acc.y));
            acc.z = __builtin_fmaf(dc, x[U].z, __builtin_fmaf(a, y[U].z, acc.z));
            acc.w = __builtin_fmaf(dc, x[U].w, __builtin_fmaf(a, y[U].w, acc.w));
            if (to != 0) {
                float* dst = (to == 1 ? dhs + (int64_t)s * dh : to == 2 ? head : tail) + col;
                if (in) *reinterpret_cast<f32x4_any_t*>(dst) = f32x4_any_t{acc.x, acc.y, acc.z, acc.w};
                acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            add<U + 1>(me, dh, col, in, acc, x, y, dhs, head, tail);
        }
    }
};

__global__ __launch_bounds__(256) void expert_bwd_sums_kernel(const float* __restrict__ xp,
                                                              const float* __restrict__ dyb,
                                                              const int32_t* __restrict__ perm,
                                                              const int32_t* __restrict__ sorted_slot,
                                                              const int32_t* __restrict__ seg_off,
                                                              const float2* __restrict__ ac, int64_t n_pairs, int hk,
                                                              int dh, float* __restrict__ dhs,
                                                              float* __restrict__ head, float* __restrict__ tail) {
    const int lane = threadIdx.x & 63;
    const int64_t n_blocks = (n_pairs + kBwdBlock - 1) / kBwdBlock;
    const int slices = (dh + kSumSlice - 1) / kSumSlice;
    const int slice = blockIdx.x % slices;
    const int col0 = slice * kSumSlice + 4 * (lane & 15);
    const bool in = col0 < dh;
    const int col = in ? col0 : 0;  // past the row: column 0, not stored
    // this quarter wave's block of positions; quarters past the last one idle with no positions
    const int64_t blk = ((int64_t)(blockIdx.x / slices) * 4 + (threadIdx.x >> 6)) * 4 + (lane >> 4);
    const int64_t b0 = blk * kBwdBlock;
    const int cnt = blk < n_blocks ? (int)min((int64_t)kBwdBlock, n_pairs - b0) : 0;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int c = 0; c < kBwdBlock; c += 16) {
        // 16 positions, a lane each; past the block's end nothing is added or stored
        const int i = c + (lane & 15);
        SumPos me{0, 0, 0, 0.0f, 0.0f};
        if (i < cnt) {
            const int p = perm[b0 + i];
            me.s = sorted_slot[b0 + i];
            const int after = i + 1 < cnt ? sorted_slot[b0 + i + 1] : -1;
            const float2 v = ac[p];
            me.t = p / hk;
            me.a = v.x;
            me.dc = v.y;
            if (after != me.s)
                me.to = seg_off[me.s] < b0 ? 2 : seg_off[me.s + 1] > b0 + kBwdBlock ? 3 : 1;
        }
        SumStep<0>::run(me, xp, dyb, dh, col, in, acc, dhs, head + blk * dh, tail + blk * dh);
        SumStep<8>::run(me, xp, dyb, dh, col, in, acc, dhs, head + blk * dh, tail + blk * dh);
    }
}

// dh of each segment that crosses blocks: found from its first block (the segment of the
// block's last position, when it began in the block and continues past it), summed over
// that block's tail part and the head parts of the blocks it continues into, in order.
template <int NB>
__global__ __launch_bounds__(256) void expert_bwd_join_kernel(const int32_t* __restrict__ sorted_slot,
                                                              const int32_t* __restrict__ seg_off, int64_t n_pairs,
                                                              int dh, const float* __restrict__ head,
                                                              const float* __restrict__ tail,
                                                              float* __restrict__ dhs) {
    const int lane = threadIdx.x & 63;
    const int64_t n_blocks = (n_pairs + kBwdBlock - 1) / kBwdBlock;
    const int64_t wave_id = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n_waves = (int64_t)gridDim.x * 4;
    for (int64_t blk = wave_id; blk < n_blocks; blk += n_waves) {
        const int64_t b0 = blk * kBwdBlock, last = b0 + kBwdBlock - 1;
        if (last >= n_pairs) continue;  // the final block has no segment continuing past it
        const int s = sorted_slot[last];
        const int64_t beg = seg_off[s], end = seg_off[s + 1];
        if (beg < b0 || end <= last + 1) continue;  // not a segment that begins here and crosses
        float acc[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int e = 64 * j + lane;
            acc[j] = e < dh ? tail[blk * dh + e] : 0.0f;
        }
        const int64_t b_end = (end - 1) / kBwdBlock;  // the segment's last block
        for (int64_t b = blk + 1; b <= b_end; ++b) {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int e = 64 * j + lane;
                if (e < dh) acc[j] += head[b * dh + e];
            }
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int e = 64 * j + lane;
            if (e < dh) dhs[(int64_t)s * dh + e] = acc[j];
        }
    }
}

size_t expert_backward_workspace_bytes(int64_t n_pairs, int dh) {
    const int64_t n_blocks = (n_pairs + kBwdBlock - 1) / kBwdBlock;
    return (size_t)n_pairs * sizeof(float2) + 2 * (size_t)n_blocks * dh * sizeof(float) + 256;
}

template <typename T, int CH>
static void launch_bwd_t(const void* hid, const float* xp, const float* dyb, const int32_t* pair_slot,
                         const void* gates, int64_t n_tok, int hk, int dh, float* dg, float* hacc, float* dxp,
                         float2* ac, int num_cus, hipStream_t stream) {
    int64_t g = (n_tok + 3) / 4;
    const int64_t cap = (int64_t)num_cus * 16;
    g = g > cap ? cap : (g < 1 ? 1 : g);
    hipLaunchKernelGGL((expert_bwd_pairs_kernel<T, CH>), dim3((unsigned)g), dim3(256), 0, stream, (const T*)hid, xp,
                       dyb, pair_slot, (const T*)gates, n_tok, hk, dh, dg, hacc, dxp, ac);
}

template <int NB>
static void launch_join_t(const int32_t* sorted_slot, const int32_t* seg_off, int64_t n_pairs, int dh, const float* head,
                          const float* tail, float* dhs, int num_cus, hipStream_t stream) {
    const int64_t n_blocks = (n_pairs + kBwdBlock - 1) / kBwdBlock;
    int64_t g = (n_blocks + 3) / 4;
    const int64_t cap = (int64_t)num_cus * 16;
    g = g > cap ? cap : (g < 1 ? 1 : g);
    hipLaunchKernelGGL((expert_bwd_join_kernel<NB>), dim3((unsigned)g), dim3(256), 0, stream, sorted_slot, seg_off,
                       n_pairs, dh, head, tail, dhs);
}

int launch_expert_backward(const void* hid, const float* xp, const float* dyb, const int32_t* pair_slot,
                           const int32_t* perm, const int32_t* sorted_slot, const int32_t* seg_off, const void* gates,
                           int64_t n_tok, int H, int k, int dh, int dtype, void* ws, float* dg, float* hacc,
                           float* dxp, float* dhs, int num_cus, hipStream_t stream) {
    const int c = apply_chunks(dh, dtype);
    const int64_t n_pairs = n_tok * H * k, n_blocks = (n_pairs + kBwdBlock - 1) / kBwdBlock;
    float2* ac = static_cast<float2*>(ws);
    float* head = reinterpret_cast<float*>(static_cast<unsigned char*>(ws) +
                                           (((size_t)n_pairs * sizeof(float2) + 255) & ~(size_t)255));
    float* tail = head + (size_t)n_blocks * dh;
    bool done = false;
#define ETHOS_BWD_CASE(TT, C)                                                                                    \
    if (!done && c <= C) {                                                                                       \
        launch_bwd_t<TT, C>(hid, xp, dyb, pair_slot, gates, n_tok, H * k, dh, dg, hacc, dxp, ac, num_cus, stream); \
        done = true;                                                                                             \
    }
    if (dtype == kBF16) {
        ETHOS_BWD_CASE(uint16_t, 1)
        ETHOS_BWD_CASE(uint16_t, 2)
        ETHOS_BWD_CASE(uint16_t, 4)
        ETHOS_BWD_CASE(uint16_t, 8)
    } else {
        ETHOS_BWD_CASE(float, 1)
        ETHOS_BWD_CASE(float, 2)
        ETHOS_BWD_CASE(float, 4)
        ETHOS_BWD_CASE(float, 8)
    }
#undef ETHOS_BWD_CASE
    if (!done) return -1;
    const int slices = (dh + kSumSlice - 1) / kSumSlice;
    hipLaunchKernelGGL(expert_bwd_sums_kernel, dim3((unsigned)((n_blocks + 15) / 16 * slices)), dim3(256), 0, stream, xp, dyb,
                       perm, sorted_slot, seg_off, (const float2*)ac, n_pairs, H * k, dh, dhs, head, tail);
    const int nb = (dh + 63) / 64;
#define ETHOS_SUMS_CASE(NBC)                                                                                      \
    if (nb <= NBC) {                                                                                              \
        launch_join_t<NBC>(sorted_slot, seg_off, n_pairs, dh, head, tail, dhs, num_cus, stream);                  \
        return (int)hipGetLastError();                                                                            \
    }
    ETHOS_SUMS_CASE(1) ETHOS_SUMS_CASE(2) ETHOS_SUMS_CASE(4) ETHOS_SUMS_CASE(8) ETHOS_SUMS_CASE(16)
    ETHOS_SUMS_CASE(32) ETHOS_SUMS_CASE(64)
#undef ETHOS_SUMS_CASE
    return -1;
}

namespace {

size_t pad256(size_t n) { return (n + 255) & ~(size_t)255; }

// Offsets in expert_grads' workspace.
struct GradsLayout {
    size_t xp, dyb, hacc, dxp, dhs, pairs, w1p, part, total;
    int split_w2, split_w1;
    bool one_pass;  // room for latent_grad.hip (which takes bf16 only)
};

GradsLayout grads_layout(int64_t n_tok, int H, int k, int64_t max_u, int dl, int dh, int d, int num_cus) {
    GradsLayout l{};
    const size_t tok = pad256((size_t)n_tok * dh * sizeof(float));
    l.xp = 0;
    l.dyb = tok;
    l.hacc = 2 * tok;
    l.dxp = 3 * tok;
    l.dhs = 4 * tok;
    l.pairs = l.dhs + pad256((size_t)max_u * dh * sizeof(float));
    l.one_pass = latent_grad_fits(max_u, dl, dh);
    l.w1p = l.pairs + pad256(expert_backward_workspace_bytes(n_tok * H * k, dh));
    l.part = l.w1p + (l.one_pass ? pad256((size_t)dh * dl * 4) : 0);
    l.split_w2 = gemm_split(dh, d, n_tok, num_cus);
    l.split_w1 = gemm_split(dh, dl, max_u, num_cus);
    const size_t p2 = l.split_w2 > 1 ? (size_t)l.split_w2 * dh * d : 0, p1 = l.split_w1 > 1 ? (size_t)l.split_w1 * dh * dl : 0;
    const size_t p0 = l.one_pass ? (size_t)latent_grad_parts(max_u, num_cus) * dh * dl : 0;
    l.total = l.part + pad256(std::max({p0, p1, p2}) * sizeof(float));
    return l;
}

}  // namespace

size_t expert_grads_workspace_bytes(int64_t n_tok, int H, int k, int64_t max_u, int dl, int dh, int d, int num_cus) {
    return grads_layout(n_tok, H, k, max_u, dl, dh, d, num_cus).total;
}

// The expert stages' backward.  Every matrix product keeps float32 sums and no less than
// float32 operands (gemm.hip), and the number of unique experts stays on the device: the
// products over the experts' rows read it there, so the host does not wait for the routing.
// 4,096 tokens, 200,070 experts, bf16: about 4.0 ms as library float32 GEMMs with the GELU
// derivative as a chain of elementwise passes over [U, d_hidden], 0.83 ms as here (d latents and
// d W1 in one pass 338 us, expert sums 173, pairs 95, d W2 83, the token products 105).
int launch_expert_grads(const void* x, const void* dy, const void* hid, const void* latents, const void* w1, const void* w2,
                        const int32_t* uniq, const int32_t* seg_off, const int32_t* n_unique, int64_t max_u,
                        const int32_t* perm, const int32_t* sorted_slot, const int32_t* pair_slot, const void* gates,
                        int64_t n_tok, int H, int k, int dl, int dh, int d, int dtype, void* ws, void* dx, float* dg,
                        void* dlat, void* dw1, void* dw2, int num_cus, hipStream_t stream) {
    const bool bf = dtype == kBF16;
    const size_t size = bf ? 2 : 4;
    const GradsLayout l = grads_layout(n_tok, H, k, max_u, dl, dh, d, num_cus);
    unsigned char* w = static_cast<unsigned char*>(ws);
    float *xp = (float*)(w + l.xp), *dyb = (float*)(w + l.dyb), *hacc = (float*)(w + l.hacc), *dxp = (float*)(w + l.dxp);
    float *dhs = (float*)(w + l.dhs), *part = (float*)(w + l.part);
    const void* w2v = (const unsigned char*)w2 + (size_t)d * dh * size;  // W_v^T
    const float inv_h = 1.0f / (float)H;
    int rc;

    Gemm g;  // xp = x W_u
    g.a = x, g.lda = d, g.b = w2, g.ldb = dh, g.c = xp, g.ldc = dh;
    g.m = n_tok, g.n = dh, g.k = d;
    if ((rc = launch_gemm(bf ? kGemmBK_BR : kGemmFK_FR, g, num_cus, stream))) return rc;
    g.a = dy, g.b = w2v, g.c = dyb, g.alpha = inv_h;  // dYB = (dy / H) W_v^T
    if ((rc = launch_gemm(bf ? kGemmBK_BR : kGemmFK_FR, g, num_cus, stream))) return rc;

    rc = launch_expert_backward(hid, xp, dyb, pair_slot, perm, sorted_slot, seg_off, gates, n_tok, H, k, dh, dtype,
                                w + l.pairs, dg, hacc, dxp, dhs, num_cus, stream);
    if (rc) return rc;

    g = Gemm{};  // d W_u^T = x^T dxp and d W_v^T = (dy / H)^T hacc, stored [d][d_hidden]
    g.a = dxp, g.lda = dh, g.b = x, g.ldb = d, g.c = dw2, g.ldc = dh;
    g.m = dh, g.n = d, g.k = n_tok;
    g.transposed = true, g.out_bf16 = bf, g.split = l.split_w2, g.part = part;
    if ((rc = launch_gemm(bf ? kGemmFR_BR : kGemmFR_FR, g, num_cus, stream))) return rc;
    g.a = hacc, g.b = dy, g.c = (unsigned char*)dw2 + (size_t)d * dh * size, g.alpha = inv_h;
    if ((rc = launch_gemm(bf ? kGemmFR_BR : kGemmFR_FR, g, num_cus, stream))) return rc;

    g = Gemm{};  // dx = dxp W_u^T
    g.a = dxp, g.lda = dh, g.b = w2, g.ldb = dh, g.c = dx, g.ldc = d;
    g.m = n_tok, g.n = d, g.k = dh, g.out_bf16 = bf;
    if ((rc = launch_gemm(bf ? kGemmFK_BK : kGemmFK_FK, g, num_cus, stream))) return rc;

    if (bf && l.one_pass)
        return launch_latent_grad(dhs, latents, w1, uniq, n_unique, max_u, dh, w + l.w1p, part, dlat, dw1, num_cus, stream);

    g = Gemm{};  // dpre = gelu'(z W1) dh, in place of dh
    g.a = latents, g.lda = dl, g.a_rows = uniq, g.b = w1, g.ldb = dl, g.c = dhs, g.ldc = dh;
    g.m = max_u, g.n = dh, g.k = dl, g.dyn = n_unique, g.epilogue = kGemmGeluGrad;
    if ((rc = launch_gemm(bf ? kGemmBK_BK : kGemmFK_FK, g, num_cus, stream))) return rc;

    g = Gemm{};  // d latents: dpre W1^T into the unique experts' rows
    g.a = dhs, g.lda = dh, g.b = w1, g.ldb = dl, g.c = dlat, g.ldc = dl, g.c_rows = uniq;
    g.m = max_u, g.n = dl, g.k = dh, g.dyn = n_unique, g.out_bf16 = bf;
    if ((rc = launch_gemm(bf ? kGemmFK_BR : kGemmFK_FR, g, num_cus, stream))) return rc;

    g = Gemm{};  // d W1 = dpre^T z
    g.a = dhs, g.lda = dh, g.b = latents, g.ldb = dl, g.b_rows = uniq, g.c = dw1, g.ldc = dl;
    g.m = dh, g.n = dl, g.k = max_u, g.dyn = n_unique, g.dyn_k = true, g.out_bf16 = bf;
    g.split = l.split_w1, g.part = part;
    return launch_gemm(bf ? kGemmFR_BR : kGemmFR_FR, g, num_cus, stream);
}

}  // namespace ethos
