// Elementwise and row kernels of the language model's blocks: RMSNorm (model.py:19-30) and the
// SwiGLU product (model.py:257-265).  Each is one pass over its operands, with the rounding
// points of the torch operations it stands for; bound by memory (or, at the small sizes of a
// decode step, by the launch).  4,113 rows: a norm of 1,024 columns 6.7 us (four torch kernels,
// 25 us), the product of 4,096 columns 23 us, 4.4 TB/s (three kernels, 62 us).
#include "ethos_common.hpp"
#include "ethos_launch.hpp"
#include "ethos_rows.hpp"

namespace ethos {
namespace {

// y = RN_T(w RN_T(x / sqrt(mean(x^2) + eps))), one wave per row, CH pieces of 16 bytes per lane in
// registers, the row read once.  Rows of x are ldx apart.
template <typename T, int CH>
__global__ __launch_bounds__(256) void rms_norm_kernel(const T* __restrict__ x, int64_t ldx, const T* __restrict__ w, int64_t rows,
                                                       int d, float eps, T* __restrict__ y) {
    constexpr int N = Vec16<T>::kN;
    typedef typename Vec16<T>::raw Raw;
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (r >= rows) return;
    Raw xr[CH], wr[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e = (c * 64 + lane) * N;
        xr[c] = *reinterpret_cast<const Raw*>(x + r * ldx + (e < d ? e : 0));
        wr[c] = *reinterpret_cast<const Raw*>(w + (e < d ? e : 0));
    }
    float f[CH][N], s = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        Vec16<T>::unpack(xr[c], f[c]);
        const bool in = (c * 64 + lane) * N < d;
#pragma unroll
        for (int v = 0; v < N; ++v) s = __builtin_fmaf(in ? f[c][v] : 0.0f, f[c][v], s);
    }
    const float k = 1.0f / sqrtf(wave_sum(s) / (float)d + eps);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e = (c * 64 + lane) * N;
        float g[N];
        Vec16<T>::unpack(wr[c], g);
#pragma unroll
        for (int v = 0; v < N; ++v) g[v] *= Elem<T>::round32(f[c][v] * k);
        if (e < d) *reinterpret_cast<Raw*>(y + r * d + e) = Vec16<T>::pack(g);
    }
}

// out [rows, d] = RN_T(RN_T(gate sigmoid(gate)) up), gate and up the halves of a row [2 d].
template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const T* __restrict__ gu, int64_t rows, int d, T* __restrict__ out) {
    constexpr int N = Vec16<T>::kN;
    typedef typename Vec16<T>::raw Raw;
    const int pieces = d / N;
    const int64_t total = rows * pieces;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / pieces;
        const int e = (int)(i - r * pieces) * N;
        const Raw a = *reinterpret_cast<const Raw*>(gu + r * 2 * d + e), b = *reinterpret_cast<const Raw*>(gu + r * 2 * d + d + e);
        float g[N], u[N];
        Vec16<T>::unpack(a, g);
        Vec16<T>::unpack(b, u);
#pragma unroll
        for (int v = 0; v < N; ++v) u[v] *= Elem<T>::round32(g[v] / (1.0f + expf(-g[v])));
        *reinterpret_cast<Raw*>(out + r * d + e) = Vec16<T>::pack(u);
    }
}

template <typename T>
int rms_norm_t(const T* x, int64_t ldx, const T* w, int64_t rows, int d, float eps, T* y, hipStream_t stream) {
    const dim3 grid((unsigned)((rows + 3) / 4));
    const int ch = (d + 64 * Vec16<T>::kN - 1) / (64 * Vec16<T>::kN);
#define ETHOS_NORM(C)                                                                                                    \
    if (ch <= C) {                                                                                                       \
        hipLaunchKernelGGL((rms_norm_kernel<T, C>), grid, dim3(256), 0, stream, x, ldx, w, rows, d, eps, y);             \
        return (int)hipGetLastError();                                                                                   \
    }
    ETHOS_NORM(1) ETHOS_NORM(2) ETHOS_NORM(4) ETHOS_NORM(8)
#undef ETHOS_NORM
    return -1;
}

}  // namespace

int launch_rms_norm(const void* x, int64_t ldx, const void* w, int64_t rows, int d, float eps, int dtype, void* y,
                    hipStream_t stream) {
    return dtype == kBF16 ? rms_norm_t((const uint16_t*)x, ldx, (const uint16_t*)w, rows, d, eps, (uint16_t*)y, stream)
                          : rms_norm_t((const float*)x, ldx, (const float*)w, rows, d, eps, (float*)y, stream);
}

int launch_swiglu(const void* gu, int64_t rows, int d, int dtype, void* out, int num_cus, hipStream_t stream) {
    const int64_t items = rows * (d / (dtype == kBF16 ? 8 : 4));
    int64_t b = (items + 255) / 256;
    const int64_t cap = (int64_t)num_cus * 32;
    b = b < cap ? b : cap;
    if (dtype == kBF16)
        hipLaunchKernelGGL((swiglu_kernel<uint16_t>), dim3((unsigned)b), dim3(256), 0, stream, (const uint16_t*)gu, rows, d,
                           (uint16_t*)out);
    else
        hipLaunchKernelGGL((swiglu_kernel<float>), dim3((unsigned)b), dim3(256), 0, stream, (const float*)gu, rows, d, (float*)out);
    return (int)hipGetLastError();
}

}  // namespace ethos
