// Tiles of float64 dot products in index order (the projections whose sums are float64 chains).
#pragma once

#include "ethos_common.hpp"

namespace ethos {

// Edge of the output tile: 64, or 32 when tiles of 64 would leave CUs without one.  The float32
// query projection of 256 tokens x 1,024 columns x 256 ran 64 tiles of 64 in 52 us, 256 tiles of
// 32 take 17; the token projection (512 columns) 49 -> 15.  At 4,096 tokens tiles
// of 32 read LDS twice as often per product.
inline int dot64_tile_edge(int64_t rows, int64_t cols, int num_cus) {
    return ((rows + 63) / 64) * ((cols + 63) / 64) >= num_cus ? 64 : 32;
}

// acc[i][j] += sum over k, in order, of x[t0 + V ty + i][k] w[c0 + V tx + j][k] for the calling
// thread's V x V of an E x E tile (V = E / 16, tx = threadIdx.x % 16, ty = threadIdx.x / 16), 256
// threads.  x is [n][d]; w [m][d], or (WR) [d][m].  The next 32 k of both operands are loaded
// into registers while the current ones are multiplied out of LDS.
template <typename T, int E, bool WR>
__device__ __forceinline__ void dot64_tile(const T* __restrict__ x, const T* __restrict__ w, int t0, int n, int c0, int m, int d,
                                           double (&acc)[E / 16][E / 16]) {
    constexpr int KC = 32, V = E / 16, N = E * KC / 256;
    // rows two doubles longer: the transposing stores of consecutive k meet two lanes a bank, and
    // the V values of a thread stay 16-byte aligned
    __shared__ __align__(16) double xs[KC][E + 2];
    __shared__ __align__(16) double ws[KC][E + 2];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    T px[N], pw[N];
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int e = tid + i * 256, r = e / KC, kk = e % KC;
            const int t = t0 + r < n ? t0 + r : n - 1, k = k0 + kk < d ? k0 + kk : d - 1;
            px[i] = x[(int64_t)t * d + k];
            if (WR) {
                const int kr = k0 + e / E < d ? k0 + e / E : d - 1, c = c0 + e % E < m ? c0 + e % E : m - 1;
                pw[i] = w[(int64_t)kr * m + c];
            } else {
                const int c = c0 + r < m ? c0 + r : m - 1;
                pw[i] = w[(int64_t)c * d + k];
            }
        }
    };
    load(0);
    for (int k0 = 0; k0 < d; k0 += KC) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int e = tid + i * 256;
            xs[e % KC][e / KC] = Elem<T>::to_f64(px[i]);
            if (WR) ws[e / E][e % E] = Elem<T>::to_f64(pw[i]);
            else ws[e % KC][e / KC] = Elem<T>::to_f64(pw[i]);
        }
        __syncthreads();
        if (k0 + KC < d) load(k0 + KC);
        const int kc = d - k0 < KC ? d - k0 : KC;
#pragma unroll 4
        for (int kk = 0; kk < kc; ++kk) {
            double a[V], b[V];
#pragma unroll
            for (int i = 0; i < V; ++i) a[i] = xs[kk][ty * V + i];
#pragma unroll
            for (int j = 0; j < V; ++j) b[j] = ws[kk][tx * V + j];
#pragma unroll
            for (int i = 0; i < V; ++i)
#pragma unroll
                for (int j = 0; j < V; ++j) acc[i][j] = fma(a[i], b[j], acc[i][j]);
        }
    }
}

}  // namespace ethos
