// Latent attention of the language model's blocks (model.py:79-165): causal softmax attention
// whose keys are each head's 64 up-projected columns followed by one rotary key that all heads
// share, and whose values are 64 wide.  Queries, keys and values are read where the projections
// left them; neither the keys nor zero-padded values are assembled in memory.
//
// rope_kernel rotates the shared key once and leaves the positions' cosines and sines (rounded
// to bf16, as the rotation uses them) for the attention kernel, which rotates each query as it
// loads it.
//
// mla_attention_kernel: one workgroup of WAVES waves per (sequence, head, 32 WAVES queries),
// keys in steps of 64 through LDS, the next step's rows in registers meanwhile.  A wave keeps
// its 32 queries in registers as the B operand of S^T = K Q^T, so that a lane holds scores of one
// query only: the running maximum, sum and rescaling are per lane (one exchange between the
// wave's halves), and the exponentials are already the B operand of O^T = V^T P^T: the sums over
// keys take the keys in the order the scores lie in, and V^T is laid out in LDS in that order.
// Scores, maxima and sums are float32; the exponentials enter the second product as bf16.
// What bounds it: a step's latency (loads, two barriers, a chain of score, exponential and value
// products) rather than the MFMAs; workgroups take the longest rows first.
// 3 x 1,371 tokens, 16 heads (17 GFLOP): 46 us and 4 for the rotations, against 219 us for the
// library's fused attention on values padded to 128 columns and about 110 us of torch operations
// that rotated, padded and laid out its operands; the same error against float64 (2.0e-3).
// 1 x 1,024 tokens (workgroups of 64 queries): 32 us against 54.
//
// The running maximum's scaled form is a product rounded by itself, also where it is subtracted:
// fused multiply-adds are written out.
#pragma clang fp contract(off)

#include "ethos_common.hpp"
#include "ethos_launch.hpp"
#include "ethos_mfma.hpp"

namespace ethos {
namespace {

constexpr int kNope = 64, kRope = 64, kVal = 64, kQk = kNope + kRope;
constexpr int kKeys = 64;  // keys per step

__device__ __forceinline__ float bf_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf_hi(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }

// [a, b] -> [a c - b s, b c + a s] on packed pairs, each product and sum rounded to bf16.
__device__ __forceinline__ void rotate2(uint32_t& a, uint32_t& b, uint32_t c, uint32_t s) {
    const uint32_t ac = pack_bf16x2(bf_lo(a) * bf_lo(c), bf_hi(a) * bf_hi(c));
    const uint32_t bs = pack_bf16x2(bf_lo(b) * bf_lo(s), bf_hi(b) * bf_hi(s));
    const uint32_t bc = pack_bf16x2(bf_lo(b) * bf_lo(c), bf_hi(b) * bf_hi(c));
    const uint32_t as = pack_bf16x2(bf_lo(a) * bf_lo(s), bf_hi(a) * bf_hi(s));
    a = pack_bf16x2(bf_lo(ac) - bf_lo(bs), bf_hi(ac) - bf_hi(bs));
    b = pack_bf16x2(bf_lo(bc) + bf_lo(as), bf_hi(bc) + bf_hi(as));
}

// k_rot rows (stride ld) of n_seq sequences of n tokens -> rotated rows kr [n_seq n][64]; the
// first sequence's threads also write cos | sin [n][32 | 32].  16 lanes a row, two angles each.
__global__ __launch_bounds__(256) void rope_kernel(const uint16_t* __restrict__ k_rot, int64_t ld, const int64_t* __restrict__ pos,
                                                   const float* __restrict__ rate, int64_t rows, int n,
                                                   uint16_t* __restrict__ kr, uint16_t* __restrict__ cs) {
    const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (row >= rows) return;
    const int i = (threadIdx.x & 15) * 2;
    const int t = (int)(row % n);
    const float p = (float)pos[t];
    const float a0 = p * rate[i], a1 = p * rate[i + 1];
    const uint32_t c = pack_bf16x2(cosf(a0), cosf(a1)), s = pack_bf16x2(sinf(a0), sinf(a1));
    uint32_t a = *reinterpret_cast<const uint32_t*>(k_rot + row * ld + i);
    uint32_t b = *reinterpret_cast<const uint32_t*>(k_rot + row * ld + 32 + i);
    rotate2(a, b, c, s);
    *reinterpret_cast<uint32_t*>(kr + row * kRope + i) = a;
    *reinterpret_cast<uint32_t*>(kr + row * kRope + 32 + i) = b;
    if (row < n) {
        *reinterpret_cast<uint32_t*>(cs + (int64_t)t * 64 + i) = c;
        *reinterpret_cast<uint32_t*>(cs + (int64_t)t * 64 + 32 + i) = s;
    }
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
union Frag {
    u32x4_t u;
    uint32_t w[4];
    bf16x8_t f;
};

template <int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void mla_attention_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kv,
                                                                      const uint16_t* __restrict__ kr,
                                                                      const uint16_t* __restrict__ cs, int n, int H, int n_bh,
                                                                      int q_tiles, float scale2, uint16_t* __restrict__ out) {
    constexpr int T = WAVES * 64;
    constexpr int KN = kKeys * 16 / T;  // 16-byte key pieces per thread
    constexpr int VN = 256 / T;         // (two value columns, eight keys) units per thread
    __shared__ __align__(16) uint16_t ks[kKeys * kQk];   // [key][dim], piece at c ^ (key % 16)
    __shared__ __align__(16) uint16_t vs[kVal * kKeys];  // [column][key slot], piece at c ^ (column / 2 % 8)
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bh = blockIdx.x % n_bh, qt = q_tiles - 1 - blockIdx.x / n_bh;
    const int h = bh % H;
    const int64_t row0 = (int64_t)(bh / H) * n;  // the sequence's first row
    const int q0 = qt * 32 * WAVES, wq0 = q0 + wave * 32;
    const int my_q = wq0 + (lane & 31);
    const int qc = my_q < n ? my_q : n - 1;

    // this lane's query: dims 16 s + 8 half + 0..7 of step s, the rotary ones rotated
    Frag fq[8];
    {
        const uint16_t* qp = q + ((row0 + qc) * H + h) * kQk + 8 * half;
#pragma unroll
        for (int s = 0; s < 8; ++s) fq[s].u = *reinterpret_cast<const u32x4_t*>(qp + 16 * s);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Frag c, sn;
            c.u = *reinterpret_cast<const u32x4_t*>(cs + (int64_t)qc * 64 + 16 * s + 8 * half);
            sn.u = *reinterpret_cast<const u32x4_t*>(cs + (int64_t)qc * 64 + 32 + 16 * s + 8 * half);
#pragma unroll
            for (int j = 0; j < 4; ++j) rotate2(fq[4 + s].w[j], fq[6 + s].w[j], c.w[j], sn.w[j]);
        }
    }

    u32x4_t kreg[KN];
    uint32_t vreg[VN][8];
    auto load = [&](int key0) {
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            const int u = tid + i * T, c = u & 15;
            const int key = key0 + (u >> 4) < n ? key0 + (u >> 4) : n - 1;
            const int64_t r = row0 + key;
            const uint16_t* p = c < 8 ? kv + (r * H + h) * (kNope + kVal) + c * 8 : kr + r * kRope + (c - 8) * 8;
            kreg[i] = *reinterpret_cast<const u32x4_t*>(p);
        }
#pragma unroll
        for (int i = 0; i < VN; ++i) {
            const int u = tid + i * T, c = u >> 5;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int kk = key0 + 16 * (c >> 1) + 8 * (j >> 2) + 4 * (c & 1) + (j & 3);
                const int key = kk < n ? kk : n - 1;
                vreg[i][j] = *reinterpret_cast<const uint32_t*>(kv + ((row0 + key) * H + h) * (kNope + kVal) + kNope + 2 * (u & 31));
            }
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            const int u = tid + i * T, c = u & 15, key = u >> 4;
            *reinterpret_cast<u32x4_t*>(ks + key * kQk + ((c ^ (key & 15)) * 8)) = kreg[i];
        }
#pragma unroll
        for (int i = 0; i < VN; ++i) {
            const int u = tid + i * T, c = u >> 5, v = 2 * (u & 31);
            const uint32_t* x = vreg[i];
            const uint4 lo = make_uint4(__builtin_amdgcn_perm(x[1], x[0], 0x05040100u), __builtin_amdgcn_perm(x[3], x[2], 0x05040100u),
                                        __builtin_amdgcn_perm(x[5], x[4], 0x05040100u), __builtin_amdgcn_perm(x[7], x[6], 0x05040100u));
            const uint4 hi = make_uint4(__builtin_amdgcn_perm(x[1], x[0], 0x07060302u), __builtin_amdgcn_perm(x[3], x[2], 0x07060302u),
                                        __builtin_amdgcn_perm(x[5], x[4], 0x07060302u), __builtin_amdgcn_perm(x[7], x[6], 0x07060302u));
            const int slot = (c ^ ((v >> 1) & 7)) * 8;
            *reinterpret_cast<uint4*>(vs + v * kKeys + slot) = lo;
            *reinterpret_cast<uint4*>(vs + (v + 1) * kKeys + slot) = hi;
        }
    };

    f32x16_t o[2] = {f32x16_zero(), f32x16_zero()};
    // the running maximum (from a finite start: scores that have overflowed to -inf weigh nothing,
    // rather than NaN) and its scaled, rounded form, which every exponential is relative to
    float m = -0x1p126f, shift = m * scale2, l = 0.0f;
    const int q_last = q0 + 32 * WAVES - 1 < n ? q0 + 32 * WAVES - 1 : n - 1;
    load(0);
    for (int key0 = 0; key0 <= q_last; key0 += kKeys) {
        store();
        __syncthreads();
        if (key0 + kKeys <= q_last) load(key0 + kKeys);
        if (key0 <= wq0 + 31) {
            f32x16_t s[2] = {f32x16_zero(), f32x16_zero()};
#pragma unroll
            for (int t = 0; t < 8; ++t) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int key = 32 * k + (lane & 31);
                    const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(ks + key * kQk + (((2 * t + half) ^ (key & 15)) * 8));
                    s[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, fq[t].f, s[k], 0, 0, 0);
                }
            }
            if (key0 + kKeys - 1 > wq0) {  // a key past the wave's first query, or past the sequence
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        s[k][i] = key0 + 32 * k + mfma32_row(i, lane) > my_q ? -INFINITY : s[k][i];
            }
            float top = s[0][0];
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int i = 0; i < 16; ++i) top = fmaxf(top, s[k][i]);
            top = fmaxf(top, __shfl_xor(top, 32, 64));
            m = fmaxf(m, top);
            const float r = __builtin_amdgcn_exp2f(shift - m * scale2);
            shift = m * scale2;
            l *= r;
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[k][i] *= r;
            Frag p[4];
            float sum = 0.0f;
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[k][i], scale2, -shift));
                    const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[k][i + 1], scale2, -shift));
                    sum += e0 + e1;
                    p[2 * k + i / 8].w[i % 8 / 2] = pack_bf16x2(e0, e1);
                }
            l += sum;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int v = 32 * k + (lane & 31);
                    const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(vs + v * kKeys + (((2 * t + half) ^ ((v >> 1) & 7)) * 8));
                    o[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, p[t].f, o[k], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    l += __shfl_xor(l, 32, 64);
    if (my_q >= n) return;
    const float inv = 1.0f / l;
    uint16_t* op = out + ((row0 + my_q) * H + h) * kVal + 4 * half;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < 16; i += 4)
            *reinterpret_cast<uint2*>(op + 32 * k + 2 * i) =
                make_uint2(pack_bf16x2(o[k][i] * inv, o[k][i + 1] * inv), pack_bf16x2(o[k][i + 2] * inv, o[k][i + 3] * inv));
}

}  // namespace

bool mla_attention_supported(int nope, int rope, int v_dim) { return nope == kNope && rope == kRope && v_dim == kVal; }

size_t mla_attention_workspace_bytes(int64_t n_seq, int64_t n) {
    return (size_t)(n_seq * n) * kRope * 2 + (((size_t)n * 64 * 2 + 255) & ~(size_t)255);
}

int launch_mla_attention(const void* q, const void* kv, const void* k_rot, int64_t k_rot_ld, const int64_t* pos, const float* rate,
                         int64_t n_seq, int64_t n, int H, float scale, void* ws, void* out, int num_cus, hipStream_t stream) {
    uint16_t* cs = (uint16_t*)ws;
    uint16_t* kr = (uint16_t*)((unsigned char*)ws + (((size_t)n * 64 * 2 + 255) & ~(size_t)255));
    const int64_t rows = n_seq * n;
    hipLaunchKernelGGL(rope_kernel, dim3((unsigned)((rows + 15) / 16)), dim3(256), 0, stream, (const uint16_t*)k_rot, k_rot_ld, pos,
                       rate, rows, (int)n, kr, cs);
    const int n_bh = (int)(n_seq * H);
    const float scale2 = scale * 1.44269504f;
    // 128 queries a workgroup; 64 where that leaves CUs without one
    const int64_t big = (n + 127) / 128;
    if (big * n_bh >= num_cus)
        hipLaunchKernelGGL((mla_attention_kernel<4>), dim3((unsigned)(big * n_bh)), dim3(256), 0, stream, (const uint16_t*)q,
                           (const uint16_t*)kv, (const uint16_t*)kr, (const uint16_t*)cs, (int)n, H, n_bh, (int)big, scale2,
                           (uint16_t*)out);
    else
        hipLaunchKernelGGL((mla_attention_kernel<2>), dim3((unsigned)((n + 63) / 64 * n_bh)), dim3(128), 0, stream,
                           (const uint16_t*)q, (const uint16_t*)kv, (const uint16_t*)kr, (const uint16_t*)cs, (int)n, H, n_bh,
                           (int)((n + 63) / 64), scale2, (uint16_t*)out);
    return (int)hipGetLastError();
}

}  // namespace ethos
