// Float32 matrix products (training path, float32 generator) on the bf16 matrix cores.
//
// A float32 operand is split into three bf16 values x = hi + mid + lo (8 significant bits each,
// 24 in all: exact down to 2^-110, where lo leaves bf16's range), so that its product with a bf16
// operand is three bf16 MFMAs whose products are exact in float32, and two float32 operands take
// nine.  The sums are float32, as in a float32 GEMM; the bf16 MFMAs run at 16 times the float32
// MFMAs' rate, so three of them cost a fifth of one float32 product and nine a little over half.
// Six of the nine (down to 2^-16 of the result) leave out up to 2^-22 of a product that a float32
// multiply-add keeps; all nine cost the float32 layer of 256 tokens 116 us against 113, and a
// training step of 500 tokens nothing that shows.  Tiles of 64 sum the products of the upper planes
// by themselves and add the others at the end: one rounding of the whole sum per 16 terms instead
// of nine (or three), which halves the error against float64 (float32 layer 2.3e-7 -> 1.3e-7, its
// gradients about 1.3e-6 -> 0.55e-6, library float32 products 2.5e-7 and 1.5e-6) at the same time;
// in tiles of 128 the second sums would halve the workgroups a CU holds.  A sum with an infinity in it comes out as NaN
// and is taken again as a float32 chain (the step of 4,096 tokens with one infinite output gradient,
// whose gradients are then NaN nearly everywhere: 2.3 -> 3.3 ms).
//
// What bounds it: at these shapes (n or k of 128 to 2,048) a step's loads, which are waited for
// before the step's products.  So many workgroups per CU rather than many steps in flight per
// workgroup: tiles of 128 x 128 (64 x 64 where those leave CUs idle), k in steps of 32 through
// one LDS buffer, the next step's rows loaded into registers while the current one is
// multiplied, then split and stored; four workgroups per CU.  (Two LDS buffers and two
// workgroups: d latents 230 us instead of 177 at that point; two steps in
// registers and three workgroups: 205 us.)  LDS rows are 32 k values
// (64 bytes) with their 16-byte pieces at slot piece ^ (row / 4 % 4): the 16 rows a fragment
// read touches at a time cover all 64 banks.  A row-wise operand ([k][m]) is transposed on the
// way: a lane takes eight k of its column, each load coalesced over the lanes.
// Measured: d W1 (512 x 128, k = 200,070) 130 us, 3.7 TB/s; d latents (200,070 x 128, k = 512)
// 158 us, 2.9 TB/s; the library's float32 GEMMs took 379 us each.
#include "ethos_common.hpp"
#include "ethos_gelu.hpp"
#include "ethos_gemm.hpp"
#include "ethos_mfma.hpp"
#include "ethos_split.hpp"

namespace ethos {
namespace {

constexpr int kGemmK = 32;      // reduction step
constexpr int kGemmThreads = 256;

// 16-byte piece `c` of LDS row `row`, in bf16 elements.
__device__ __forceinline__ int lds_slot(int row, int c) { return (row * 4 + (c ^ ((row >> 2) & 3))) * 8; }

// One operand's tile of ROWS rows by kGemmK: its loads into registers and its stores into LDS.
// KC: k contiguous, else k is the row; IDX: rows taken through an index array.  A step that ends
// inside the tile takes the loads' checked form (zeros past the end), the others none.
template <typename T, bool KC, bool IDX, int ROWS> struct Tile;

template <typename T> struct Planes { static constexpr int kN = 3; };
template <> struct Planes<uint16_t> { static constexpr int kN = 1; };

__device__ __forceinline__ void put8(uint16_t* lds, int rows, int slot, const float* v) {
    uint4 p[3];
    split3(v[0], v[1], p[0].x, p[1].x, p[2].x);
    split3(v[2], v[3], p[0].y, p[1].y, p[2].y);
    split3(v[4], v[5], p[0].z, p[1].z, p[2].z);
    split3(v[6], v[7], p[0].w, p[1].w, p[2].w);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(lds + i * rows * kGemmK + slot) = p[i];
}

// k contiguous: a thread takes 8 k (32 or 16 bytes) of a row.
template <typename T, bool IDX, int ROWS> struct Tile<T, true, IDX, ROWS> {
    static constexpr int N = ROWS * 4 / kGemmThreads;
    static constexpr int W = sizeof(T) / 2;  // 16-byte loads per piece
    const T* src[N];
    uint4 v[N][W];
    bool ok[N];  // IDX: the index is a row
    __device__ __forceinline__ void init(const void* base, int64_t ld, const int32_t* rows, int64_t limit, int64_t row0,
                                         int64_t n_rows, int64_t k0, int tid) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = tid + i * kGemmThreads;
            int64_t r = row0 + (q >> 2);
            r = r < n_rows ? r : n_rows - 1;
            if (IDX) r = rows[r];
            ok[i] = !IDX || (r >= 0 && r < limit);
            r = ok[i] ? r : 0;
            src[i] = (const T*)base + r * ld + k0 + (q & 3) * 8;
        }
    }
    __device__ __forceinline__ void load(int left, int tid) {  // left: k from this step's first to the end
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int c = (tid + i * kGemmThreads) & 3;
            const bool in = c * 8 < left;
            const uint4* p = reinterpret_cast<const uint4*>(in ? src[i] : src[i] - c * 8);
#pragma unroll
            for (int w = 0; w < W; ++w) v[i][w] = p[w];
            src[i] += kGemmK;
        }
        if (IDX || left < kGemmK) {
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (!ok[i] || ((tid + i * kGemmThreads) & 3) * 8 >= left)
#pragma unroll
                    for (int w = 0; w < W; ++w) v[i][w] = make_uint4(0, 0, 0, 0);
        }
    }
    __device__ __forceinline__ void store(uint16_t* lds, int tid) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = tid + i * kGemmThreads;
            if constexpr (W == 2) {
                const float f[8] = {__uint_as_float(v[i][0].x), __uint_as_float(v[i][0].y), __uint_as_float(v[i][0].z),
                                    __uint_as_float(v[i][0].w), __uint_as_float(v[i][1].x), __uint_as_float(v[i][1].y),
                                    __uint_as_float(v[i][1].z), __uint_as_float(v[i][1].w)};
                put8(lds, ROWS, lds_slot(q >> 2, q & 3), f);
            } else {
                *reinterpret_cast<uint4*>(lds + lds_slot(q >> 2, q & 3)) = v[i][0];
            }
        }
    }
};

// k as the row: a thread takes eight k of one column (bf16 tiles of 128: of two adjacent
// columns, one 4-byte load for both; in a tile of 64 that would leave half the threads idle).
template <typename T, bool IDX, int ROWS> struct Tile<T, false, IDX, ROWS> {
    static constexpr bool kPair = sizeof(T) == 2 && ROWS >= 128;
    static constexpr int W = kPair ? ROWS / 2 : ROWS;  // lanes' units per piece
    static constexpr int N = W * 4 / kGemmThreads;
    const T* src[N];       // (IDX: the column only) at this step's first k of the thread's piece
    const int32_t* rows;
    int64_t ld;
    uint32_t v[N][8];
    __device__ __forceinline__ void init(const void* base, int64_t l, const int32_t* rws, int64_t /*limit*/, int64_t row0,
                                         int64_t n_rows, int64_t k0, int tid) {
        ld = l;
        rows = IDX ? rws + k0 : nullptr;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = tid + i * kGemmThreads, u = q % W;
            const int64_t r = row0 + (kPair ? 2 * u : u);
            const int64_t last = kPair ? n_rows - 2 : n_rows - 1;
            const int64_t col = r < last ? r : last;
            src[i] = (const T*)base + col + (IDX ? 0 : (k0 + __builtin_amdgcn_readfirstlane(q / W) * 8) * l);
        }
    }
    __device__ __forceinline__ static uint32_t get(const T* p) {
        if constexpr (kPair || sizeof(T) == 4) return *reinterpret_cast<const uint32_t*>(p);
        else return *p;
    }
    __device__ __forceinline__ void load(int left, int tid) {
        if (left >= kGemmK) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int c = __builtin_amdgcn_readfirstlane((tid + i * kGemmThreads) / W);
                int32_t id[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) id[j] = IDX ? rows[c * 8 + j] : j;
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] = get(src[i] + id[j] * ld);
            }
        } else {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int c = __builtin_amdgcn_readfirstlane((tid + i * kGemmThreads) / W);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int k = c * 8 + j;
                    const int kk = k < left ? k : left - 1;
                    const uint32_t x = get(src[i] + (IDX ? (int64_t)rows[kk] : (int64_t)(kk - c * 8)) * ld);
                    v[i][j] = k < left ? x : 0u;
                }
            }
        }
        if (IDX) {
            rows += kGemmK;
        } else {
#pragma unroll
            for (int i = 0; i < N; ++i) src[i] += kGemmK * ld;
        }
    }
    __device__ __forceinline__ void store(uint16_t* lds, int tid) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = tid + i * kGemmThreads, u = q % W, c = q / W;
            const uint32_t* x = v[i];
            if constexpr (sizeof(T) == 4) {
                float f[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] = __uint_as_float(x[j]);
                put8(lds, ROWS, lds_slot(u, c), f);
            } else {
                const uint4 lo = make_uint4(__builtin_amdgcn_perm(x[1], x[0], 0x05040100u), __builtin_amdgcn_perm(x[3], x[2], 0x05040100u),
                                            __builtin_amdgcn_perm(x[5], x[4], 0x05040100u), __builtin_amdgcn_perm(x[7], x[6], 0x05040100u));
                *reinterpret_cast<uint4*>(lds + lds_slot(kPair ? 2 * u : u, c)) = lo;
                if constexpr (kPair) {
                    const uint4 hi = make_uint4(__builtin_amdgcn_perm(x[1], x[0], 0x07060302u), __builtin_amdgcn_perm(x[3], x[2], 0x07060302u),
                                                __builtin_amdgcn_perm(x[5], x[4], 0x07060302u), __builtin_amdgcn_perm(x[7], x[6], 0x07060302u));
                    *reinterpret_cast<uint4*>(lds + lds_slot(2 * u + 1, c)) = hi;
                }
            }
        }
    }
};

// Workgroup -> (part of the reduction, row tile, column tile).  Workgroup b runs on XCD b % 8;
// tiles that read the same rows form a group that stays on one XCD, one after the other, so that
// those rows come from memory once and then from that XCD's L2: the column tiles of a row tile,
// or, with eight or more parts, all tiles of a part.  Groups go round the XCDs (with a device
// count that cuts the rows short, every XCD loses the same share).  The grid holds whole rounds.
struct GemmGroups {
    int64_t groups;
    int each;
};
__host__ __device__ inline GemmGroups gemm_groups(int split, int64_t mt, int nt) {
    return split >= 8 ? GemmGroups{split, (int)mt * nt} : GemmGroups{split * mt, nt};
}

// The rows of C in use and one part's [kb, ke) of the reduction (all of it when not split).
struct GemmRange {
    int64_t m, kb, ke;
};
__device__ __forceinline__ GemmRange gemm_range(const Gemm& p, int part_id) {
    GemmRange r{p.m, 0, p.k};
    if (p.dyn) {
        const int64_t d = *p.dyn;
        if (p.dyn_k) r.ke = d < r.ke ? d : r.ke;
        else r.m = d < r.m ? d : r.m;
    }
    if (p.split > 1) {
        const int64_t k = r.ke, per = ((k + p.split - 1) / p.split + kGemmK - 1) / kGemmK * kGemmK;
        r.kb = per * part_id;
        r.ke = r.kb + per < k ? r.kb + per : k;
    }
    return r;
}

// One output's sum over a part of the reduction as a float32 chain: what an infinity needs, which
// against the other operand's lower planes gives NaNs (times zero) and infinities of either sign.
template <typename TA, bool AK, typename TB, bool BK, bool IDX>
__device__ __forceinline__ float gemm_chain(const Gemm& p, int64_t m, int n, int part_id) {
    const GemmRange r = gemm_range(p, part_id);
    const int64_t row = IDX && AK ? (int64_t)p.a_rows[m] : m;
    const bool zeros = IDX && AK && (row < 0 || row >= p.a_limit);
    float s = 0.0f;
    for (int64_t k = r.kb; k < r.ke && s == s; ++k) {  // (a NaN stays one)
        const int64_t kr = IDX && !BK ? (int64_t)p.b_rows[k] : k;
        const float a = zeros ? 0.0f : Elem<TA>::to_f32(((const TA*)p.a)[AK ? row * p.lda + k : k * p.lda + row]);
        const float b = Elem<TB>::to_f32(((const TB*)p.b)[BK ? (int64_t)n * p.ldb + k : kr * p.ldb + n]);
        s = __builtin_fmaf(a, b, s);
    }
    return s;
}

template <typename TA, bool AK, typename TB, bool BK, bool IDX, int BM, int BN>
__global__ __launch_bounds__(kGemmThreads, (BM > 64 ? (sizeof(TB) == 4 ? 3 : 4) : 4)) void gemm_kernel(Gemm p) {
    constexpr int PA = Planes<TA>::kN, PB = Planes<TB>::kN;
    constexpr int MI = BM / 64, NI = BN / 64;
    constexpr int kBuf = (PA * BM + PB * BN) * kGemmK;
    __shared__ __align__(16) uint16_t lds[kBuf];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt = (p.n + BN - 1) / BN;
    const int64_t mt = (p.m + BM - 1) / BM;
    const GemmGroups gg = gemm_groups(p.split, mt, nt);
    const int64_t group = (int64_t)(blockIdx.x / 8) / gg.each * 8 + blockIdx.x % 8;
    const int64_t tile = group * gg.each + (blockIdx.x / 8) % gg.each;  // (part, row tile, column tile)
    const int part_id = (int)(tile / (mt * nt));
    const int64_t m0 = tile / nt % mt * BM;
    const int n0 = (int)(tile % nt) * BN;
    const GemmRange range = gemm_range(p, part_id);
    const int64_t m = range.m, kb = range.kb, ke = range.ke;
    if (group >= gg.groups || m0 >= m) return;
    // sums of the products of upper planes, and (kApart) of the others, added at the end
    constexpr bool kApart = PA + PB > 2 && MI * NI == 1;
    f32x16_t acc[MI][NI], low = f32x16_zero();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x16_zero();

    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    if (kb < ke) {
        Tile<TA, AK, IDX && AK, BM> ta;
        Tile<TB, BK, IDX && !BK, BN> tb;
        ta.init(p.a, p.lda, p.a_rows, p.a_limit, m0, m, kb, tid);
        tb.init(p.b, p.ldb, p.b_rows, INT64_MAX, n0, p.n, kb, tid);
        int64_t left = ke - kb;
        ta.load(left < kGemmK ? (int)left : kGemmK, tid);
        tb.load(left < kGemmK ? (int)left : kGemmK, tid);
        const uint16_t* la = lds;
        const uint16_t* lb = lds + PA * BM * kGemmK;
        for (; left > 0; left -= kGemmK) {
            ta.store(lds, tid);
            tb.store(lds + PA * BM * kGemmK, tid);
            __syncthreads();
            if (left > kGemmK) {
                const int next = left - kGemmK < kGemmK ? (int)(left - kGemmK) : kGemmK;
                ta.load(next, tid);
                tb.load(next, tid);
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const int c = ks * 2 + (lane >> 5);
                bf16x8_t fa[MI][PA], fb[NI][PB];
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int q = 0; q < PA; ++q)
                        fa[i][q] = *reinterpret_cast<const bf16x8_t*>(la + q * BM * kGemmK + lds_slot(wm + i * 32 + (lane & 31), c));
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int q = 0; q < PB; ++q)
                        fb[j][q] = *reinterpret_cast<const bf16x8_t*>(lb + q * BN * kGemmK + lds_slot(wn + j * 32 + (lane & 31), c));
                // smallest products first
#pragma unroll
                for (int q = PA + PB - 2; q >= 0; --q) {
#pragma unroll
                    for (int qa = 0; qa < PA; ++qa) {
                        const int qb = q - qa;
                        if (qb < 0 || qb >= PB) continue;
#pragma unroll
                        for (int i = 0; i < MI; ++i)
#pragma unroll
                            for (int j = 0; j < NI; ++j) {
                                f32x16_t& to = kApart && q > 0 ? low : acc[i][j];
                                to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][qa], fb[j][qb], to, 0, 0, 0);
                            }
                    }
                }
            }
            __syncthreads();
        }
    }

    if constexpr (kApart) acc[0][0] += low;
    float* part = p.split > 1 ? p.part + (size_t)part_id * (size_t)p.m * (size_t)p.n : nullptr;
    auto emit = [&](int64_t mm, int n, float v, float bias, float aux) {
        if (part) {
            part[p.transposed ? (int64_t)n * p.m + mm : mm * p.n + n] = v;
            return;
        }
        const int64_t row = p.c_rows ? p.c_rows[mm] : mm;
        const int64_t at = p.transposed ? n * p.ldc + row : row * p.ldc + n;
        if (p.epilogue == kGemmGeluGrad) ((float*)p.c)[at] = gelu_erf_grad(v) * aux;
        else if (p.epilogue == kGemmGelu) ((float*)p.c)[at] = gelu_erf(v);
        else if (p.out_bf16) ((uint16_t*)p.c)[at] = f32_to_bf16_bits(__builtin_fmaf(p.alpha, v, bias));
        else ((float*)p.c)[at] = __builtin_fmaf(p.alpha, v, bias);
    };
    constexpr bool kPlanes = PA + PB > 2;
    uint64_t again = 0;  // (planes) this thread's outputs (j, i, g) that came out as NaN
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int n = n0 + wn + j * 32 + (lane & 31);
        const int nc = n < p.n ? n : p.n - 1;
        const float bias = p.bias ? Elem<TB>::to_f32(((const TB*)p.bias)[nc]) : 0.0f;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int64_t mb = m0 + wm + i * 32;
            float aux[16] = {};
            if (p.epilogue == kGemmGeluGrad) {
                // all sixteen requested before any is used
#pragma unroll
                for (int g = 0; g < 16; ++g) {
                    const int64_t mm = mb + mfma32_row(g, lane);
                    aux[g] = ((const float*)p.c)[(mm < m ? mm : m - 1) * p.ldc + nc];
                }
            }
            if (n >= p.n) continue;
#pragma unroll
            for (int g = 0; g < 16; ++g) {
                const int64_t mm = mb + mfma32_row(g, lane);
                if (mm >= m) continue;
                if (kPlanes && acc[i][j][g] != acc[i][j][g]) again |= 1ull << ((j * MI + i) * 16 + g);
                else emit(mm, n, acc[i][j][g], bias, aux[g]);
            }
        }
    }
    if constexpr (kPlanes) {
        for (; again != 0; again &= again - 1) {
            const int e = __builtin_ctzll(again), g = e & 15, i = (e >> 4) % MI, j = (e >> 4) / MI;
            const int64_t mm = m0 + wm + i * 32 + mfma32_row(g, lane);
            const int n = n0 + wn + j * 32 + (lane & 31);
            const float bias = p.bias ? Elem<TB>::to_f32(((const TB*)p.bias)[n]) : 0.0f;
            const float aux = p.epilogue == kGemmGeluGrad ? ((const float*)p.c)[mm * p.ldc + n] : 0.0f;
            emit(mm, n, gemm_chain<TA, AK, TB, BK, IDX>(p, mm, n, part_id), bias, aux);
        }
    }
}

// Sum of the split partial products, in order, and the result's form.  rows x cols as stored.
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* __restrict__ part, int split, int64_t rows,
                                                          int64_t cols, float alpha, int out_bf16,
                                                          void* __restrict__ c, int64_t ldc) {
    const int64_t n = rows * cols;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        float s = 0.0f;
        for (int z0 = 0; z0 < split; z0 += 8) {
            float v[8];
#pragma unroll
            for (int z = 0; z < 8; ++z) v[z] = part[(size_t)(z0 + z < split ? z0 + z : split - 1) * n + i];
#pragma unroll
            for (int z = 0; z < 8; ++z) s += z0 + z < split ? v[z] : 0.0f;
        }
        const int64_t at = i / cols * ldc + i % cols;
        if (out_bf16) ((uint16_t*)c)[at] = f32_to_bf16_bits(alpha * s);
        else ((float*)c)[at] = alpha * s;
    }
}

}  // namespace

int launch_gemm_reduce(const float* part, int split, int64_t rows, int64_t cols, float alpha, bool out_bf16, void* c, int64_t ldc,
                       hipStream_t stream) {
    int64_t rb = (rows * cols + 255) / 256;
    rb = rb > 4096 ? 4096 : rb;
    hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)rb), dim3(256), 0, stream, part, split, rows, cols, alpha,
                       out_bf16 ? 1 : 0, c, ldc);
    return (int)hipGetLastError();
}

namespace {

template <typename TA, bool AK, typename TB, bool BK, bool IDX, int BM, int BN>
int launch_t(const Gemm& g, hipStream_t stream) {
    const int64_t mt = (g.m + BM - 1) / BM, nt = (g.n + BN - 1) / BN;
    const GemmGroups gg = gemm_groups(g.split, mt, (int)nt);
    const int64_t blocks = (gg.groups + 7) / 8 * 8 * gg.each;
    if (blocks > INT32_MAX) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_kernel<TA, AK, TB, BK, IDX, BM, BN>), dim3((unsigned)blocks), dim3(kGemmThreads), 0,
                       stream, g);
    if (g.split > 1) {
        const int64_t rows = g.transposed ? g.n : g.m, cols = g.transposed ? g.m : g.n;
        return launch_gemm_reduce(g.part, g.split, rows, cols, g.alpha, g.out_bf16, g.c, g.ldc, stream);
    }
    return (int)hipGetLastError();
}

template <typename TA, bool AK, typename TB, bool BK>
int launch_form(const Gemm& g, int num_cus, hipStream_t stream) {
    // 128 x 128 tiles when they give every CU one, else 64 x 64
    const int64_t big = ((g.m + 127) / 128) * ((g.n + 127) / 128) * g.split;
    const bool large = big >= num_cus && g.n > 64;
    if (AK ? g.a_rows != nullptr : g.b_rows != nullptr)
        return large ? launch_t<TA, AK, TB, BK, true, 128, 128>(g, stream) : launch_t<TA, AK, TB, BK, true, 64, 64>(g, stream);
    return large ? launch_t<TA, AK, TB, BK, false, 128, 128>(g, stream) : launch_t<TA, AK, TB, BK, false, 64, 64>(g, stream);
}

}  // namespace

int gemm_split(int64_t m, int n, int64_t k, int num_cus) {
    const int64_t tiles = ((m + 127) / 128) * ((n + 127) / 128);
    int64_t s = 2 * (int64_t)num_cus / tiles;
    const int64_t most = k / 256;
    s = s < most ? s : most;
    if (s > 8) s -= s % 8;  // whole rounds of the XCDs
    return (int)(s < 1 ? 1 : s);
}

int launch_gemm(GemmForm form, const Gemm& g, int num_cus, hipStream_t stream) {
    if (g.m <= 0 || g.n <= 0) return 0;
    switch (form) {
        case kGemmBK_BK: return launch_form<uint16_t, true, uint16_t, true>(g, num_cus, stream);
        case kGemmBK_BR: return launch_form<uint16_t, true, uint16_t, false>(g, num_cus, stream);
        case kGemmFK_BK: return launch_form<float, true, uint16_t, true>(g, num_cus, stream);
        case kGemmFK_BR: return launch_form<float, true, uint16_t, false>(g, num_cus, stream);
        case kGemmFR_BR: return launch_form<float, false, uint16_t, false>(g, num_cus, stream);
        case kGemmFK_FK: return launch_form<float, true, float, true>(g, num_cus, stream);
        case kGemmFK_FR: return launch_form<float, true, float, false>(g, num_cus, stream);
        case kGemmFR_FR: return launch_form<float, false, float, false>(g, num_cus, stream);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace ethos
