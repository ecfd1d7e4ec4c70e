// The experts' part of the backward in one pass (bf16, d_latent 128): dpre = gelu'(z W1) dh,
// d latents = dpre W1^T and d W1 = dpre^T z, with dh [U][d_hidden] float32 read once and dpre
// never stored.  As three products it is written and read back twice, 2.1 GB at 200,070 experts
// of 512 hidden values, of which 0.42 are dh itself.
//
// A workgroup of eight waves walks tiles of 64 experts, 256 hidden columns a pass, a wave 32 of
// them.  Per pass:
//   1. z W1 on the matrix cores: a lane holds one hidden column of sixteen experts, times gelu'
//      and dh, split exactly into three bf16 planes (ethos_split.hpp).
//   2. d W1: those planes are the operand of dpre^T z as they lie in the registers; z's transposed
//      copy in LDS has its experts in that order.  A wave's 32 x 128 sums stay in registers for
//      all tiles (128 registers at d_hidden 512) and leave once, as this workgroup's partial sum.
//   3. d latents need the planes with the hidden columns along a lane, from LDS: neighbouring
//      lanes exchange halves first, so that the writes are whole words.  A wave takes 32 experts by
//      32 latents over the pass's 256 columns.
// One workgroup per CU (256 registers a lane, 132 KB of LDS).  What bounds it: the phases follow
// one another with a barrier between, so that per tile of 64 and SIMD about 13,000 cycles of MFMA
// and 26,000 of VALU (gelu', the splits) hardly overlap, with two waves to hide any latency.
// Measured, 200,070 experts of 512 hidden values: 318 us and 20 us to add up the workgroups' d W1,
// against 502 us as products (dpre 201, d latents 175, d W1 116 + 10); for 512 tokens' pairs 108
// and 16 against 185, for 128 tokens' (16,384 pairs) 36 and 12 against 94.
// W1's fragments are requested a phase ahead: 350 us when each was requested where it is used.
#include "ethos_common.hpp"
#include "ethos_gelu.hpp"
#include "ethos_gemm.hpp"
#include "ethos_launch.hpp"
#include "ethos_mfma.hpp"
#include "ethos_split.hpp"

namespace ethos {
namespace {

constexpr int kLgRows = 64, kLgThreads = 512, kLgDl = 128, kLgPass = 256;
constexpr int kLgPitch = kLgPass + 8;  // plane rows (bf16): a fragment's 16 rows on all banks
constexpr int kLgZn = kLgDl + 8;       // z rows

// Piece (8 experts) `q` of latent column `l` in the transposed z tile: the 16 columns that a
// fragment read touches at a time, and the 8 that a row's store does, lie on different banks.
__device__ __forceinline__ int zt_at(int l, int q) { return l * kLgRows + (q ^ (((l >> 1) ^ (l >> 3)) & 7)) * 8; }

// W1 [d_hidden][128] in the order of the two products' fragments: wf, for z W1, [d_hidden / 32]
// [8 steps of 16 latents][lane][8 latents]; wp, for d latents, [d_hidden / 8][128][8 columns].
__global__ __launch_bounds__(256) void w1_pieces_kernel(const uint16_t* __restrict__ w1, int dh, uint16_t* __restrict__ wf,
                                                        uint16_t* __restrict__ wp) {
    const int i = blockIdx.x * 256 + threadIdx.x;  // (piece of 8 hidden columns, latent) of wp
    if (i >= dh / 8 * kLgDl) return;
    const int l = i % kLgDl, h = i / kLgDl * 8;
    uint32_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = w1[(h + j) * kLgDl + l];
    const int col = i / 512 * 32 + (i & 31), l0 = (i >> 6 & 7) * 16 + (i >> 5 & 1) * 8;  // i as (block, step, lane) of wf
    *reinterpret_cast<uint4*>(wf + (size_t)i * 8) = *reinterpret_cast<const uint4*>(w1 + col * kLgDl + l0);
    *reinterpret_cast<uint4*>(wp + (size_t)i * 8) =
        make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
}

// v, but not known to the compiler to be the same each time: LDS and row addresses made from it
// are formed where they are used instead of being kept over the whole loop (about 100 registers).
__device__ __forceinline__ int fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <int P>
__global__ __launch_bounds__(kLgThreads, 2) void latent_grad_kernel(const float* __restrict__ dhs,
                                                                    const uint16_t* __restrict__ latents,
                                                                    const uint16_t* __restrict__ w1f,
                                                                    const uint16_t* __restrict__ w1p,
                                                                    const int32_t* __restrict__ uniq,
                                                                    const int32_t* __restrict__ n_unique, int64_t max_u,
                                                                    uint16_t* __restrict__ dlat, float* __restrict__ part) {
    constexpr int kDh = P * kLgPass;
    __shared__ __align__(16) uint16_t planes[3 * kLgRows * kLgPitch];
    __shared__ __align__(16) uint16_t zn[kLgRows * kLgZn];
    __shared__ __align__(16) uint16_t zt[kLgDl * kLgRows];
    __shared__ int32_t ids[2][kLgRows];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int64_t m = *n_unique;
    m = m < max_u ? m : max_u;
    const int64_t step = (int64_t)gridDim.x * kLgRows;
    int64_t m0 = (int64_t)blockIdx.x * kLgRows;

    f32x16_t acc[P][4];
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x16_zero();

    if (m0 < m) {
        // staging: eight threads a row, 16 latents each (pieces c and c + 8)
        const int e = tid >> 3;
        const int zpos = (e >> 4) * 16 + ((e >> 2) & 1) * 8 + ((e >> 3) & 1) * 4 + (e & 3);
        float d[2][16];
        // (one uniform base and 32-bit offsets: 64-bit addresses would take the registers)
        auto load_d = [&](int64_t r0, int pass) {
            const int lane = fresh(tid & 63);
            const float* base = dhs + r0 * kDh + pass * kLgPass + wave * 32;
            const int last = (int)(m - r0 < kLgRows ? m - r0 : kLgRows) - 1;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int r = 32 * t + mfma32_row(i, lane);
                    d[t][i] = base[(unsigned)((r < last ? r : last) * kDh + (lane & 31))];
                }
        };
        auto id_of = [&](int64_t r0) { return r0 + e < m ? uniq[r0 + e] : -1; };
        uint4 z[2];
        auto load_z = [&](int32_t id) {
            const uint4* p = reinterpret_cast<const uint4*>(latents + (int64_t)(id < 0 ? 0 : id) * kLgDl);
            z[0] = p[tid & 7], z[1] = p[(tid & 7) + 8];
        };
        int32_t id = id_of(m0), next_id = id_of(m0 + step);
        load_z(id);
        load_d(m0, 0);
        // W1's fragments of a pass, four steps at a time, requested a phase or a group of products
        // before their use (again for each tile)
        bf16x8_t fw[8], fp[16];
        auto load_w = [&](int pass, int k0) {
            const unsigned at = fresh(tid & 63) * 8;
#pragma unroll
            for (int ks = k0; ks < k0 + 4; ++ks)
                fw[ks] = *reinterpret_cast<const bf16x8_t*>(w1f + (pass * 8 + wave) * (32 * kLgDl) + at + ks * 512);
        };
        auto load_p = [&](int pass, int k0) {
            const int lane = fresh(tid & 63);
            const unsigned at = ((lane >> 5) * kLgDl + (wave & 3) * 32 + (lane & 31)) * 8;
#pragma unroll
            for (int ks = k0; ks < k0 + 4; ++ks)
                fp[ks] = *reinterpret_cast<const bf16x8_t*>(w1p + at + (pass * (kLgPass / 8) + ks * 2) * kLgDl * 8);
        };
        load_w(0, 0);
        int par = 0;
        for (; m0 < m; m0 += step, par ^= 1) {
            // z rows and their transposed copy (rows past the end: zeros)
            const int c = fresh(tid & 7);
            if (id < 0) z[0] = z[1] = make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int l0 = (c + 8 * q) * 8;
                *reinterpret_cast<uint4*>(zn + e * kLgZn + l0) = z[q];
                const uint32_t v[4] = {z[q].x, z[q].y, z[q].z, z[q].w};
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    zt[zt_at(l0 + j, zpos >> 3) + (zpos & 7)] = (uint16_t)(v[j >> 1] >> (16 * (j & 1)));
            }
            if (c == 0) ids[par][e] = id;
            __syncthreads();

            const int rows = (int)(m - m0 < kLgRows ? m - m0 : kLgRows);
            f32x16_t dl = f32x16_zero();
            const int te = wave >> 2, lt0 = (wave & 3) * 32;
#pragma unroll
            for (int pass = 0; pass < P; ++pass) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int lane = fresh(tid & 63), l32 = lane & 31, hf = lane >> 5;
                    f32x16_t pre = f32x16_zero();
#pragma unroll
                    for (int k0 = 0; k0 < 8; k0 += 4) {
                        if (k0 == 0) load_w(pass, 4);
                        __builtin_amdgcn_sched_barrier(0);
                        bf16x8_t fz[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            fz[u] = *reinterpret_cast<const bf16x8_t*>(zn + (32 * t + l32) * kLgZn + (k0 + u) * 16 + hf * 8);
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            pre = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fz[u], fw[k0 + u], pre, 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    uint32_t w[3][8];
#pragma unroll
                    for (int g = 0; g < 8; ++g) {
                        float v[2];
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            const int i = 2 * g + j;
                            v[j] = gelu_erf_grad(pre[i]) * d[t][i];
                            if (32 * t + mfma32_row(i, lane) >= rows) v[j] = 0.0f;
                        }
                        split3(v[0], v[1], w[0][g], w[1][g], w[2][g]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    // to LDS: even lanes take row 2 g of two columns, odd lanes row 2 g + 1
                    const uint32_t sel = lane & 1 ? 0x03020706u : 0x05040100u;
#pragma unroll
                    for (int g = 0; g < 8; ++g) {
                        const int row = 32 * t + mfma32_row(2 * g, lane) + (lane & 1);
#pragma unroll
                        for (int q = 0; q < 3; ++q) {
                            const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)w[q][g], 0xB1, 0xF, 0xF, true);
                            *reinterpret_cast<uint32_t*>(planes + (q * kLgRows + row) * kLgPitch + wave * 32 + (l32 & ~1)) =
                                __builtin_amdgcn_perm(other, w[q][g], sel);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (t == 0) load_w(pass, 0);
                    else load_p(pass, 0);
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        __builtin_amdgcn_sched_barrier(0);
                        bf16x8_t fb[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            fb[j] = *reinterpret_cast<const bf16x8_t*>(zt + zt_at(j * 32 + l32, (t * 2 + s) * 2 + hf));
#pragma unroll
                        for (int q = 2; q >= 0; --q) {  // smallest products first
                            const uint4 u = make_uint4(w[q][4 * s], w[q][4 * s + 1], w[q][4 * s + 2], w[q][4 * s + 3]);
                            const bf16x8_t fa = __builtin_bit_cast(bf16x8_t, u);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                acc[pass][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb[j], acc[pass][j], 0, 0, 0);
                        }
                    }
                }
                __syncthreads();
                const int lane = fresh(tid & 63), l32 = lane & 31, hf = lane >> 5;
                load_p(pass, 4);
                auto products = [&](int k0) {
#pragma unroll
                    for (int ks = k0; ks < k0 + 4; ++ks) {
#pragma unroll
                        for (int q = 2; q >= 0; --q)
                            dl = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                *reinterpret_cast<const bf16x8_t*>(planes + (q * kLgRows + 32 * te + l32) * kLgPitch + ks * 16 + hf * 8),
                                fp[ks], dl, 0, 0, 0);
                        if (ks % 2 == 1) __builtin_amdgcn_sched_barrier(0);
                    }
                };
                __builtin_amdgcn_sched_barrier(0);
                products(0);
                load_p(pass, 8);
                products(4);
                load_p(pass, 12);
                // the next pass's dh (its loads come back in order: after this pass's W1)
                if (pass + 1 < P) {
                    load_d(m0, pass + 1);
                } else if (m0 + step < m) {
                    load_d(m0 + step, 0);
                    id = next_id;
                    load_z(id);
                    next_id = id_of(m0 + 2 * step);
                }
                __builtin_amdgcn_sched_barrier(0);
                products(8);
                products(12);
                load_w(pass + 1 < P ? pass + 1 : 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (pass + 1 < P) __syncthreads();  // (after the last pass: the next tile's first barrier)
            }
            const int lane = fresh(tid & 63), l32 = lane & 31;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 32 * te + mfma32_row(i, lane);
                if (r < rows) dlat[(int64_t)ids[par][r] * kLgDl + lt0 + l32] = f32_to_bf16_bits(dl[i]);
            }
        }
    }
    const int lane = tid & 63, l32 = lane & 31;
    float* out = part + (size_t)blockIdx.x * kDh * kLgDl;
#pragma unroll
    for (int pass = 0; pass < P; ++pass)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                out[(pass * kLgPass + wave * 32 + mfma32_row(i, lane)) * kLgDl + j * 32 + l32] = acc[pass][j][i];
}

}  // namespace

bool latent_grad_fits(int64_t max_u, int dl, int dh) {
    return dl == kLgDl && (dh == kLgPass || dh == 2 * kLgPass) && max_u >= kLatentGradRows;
}

int latent_grad_parts(int64_t max_u, int num_cus) {
    const int64_t tiles = (max_u + kLgRows - 1) / kLgRows;
    return (int)(tiles < num_cus ? tiles : num_cus);
}

int launch_latent_grad(const float* dhs, const void* latents, const void* w1, const int32_t* uniq, const int32_t* n_unique,
                       int64_t max_u, int dh, void* w1p, float* part, void* dlat, void* dw1, int num_cus, hipStream_t stream) {
    const int parts = latent_grad_parts(max_u, num_cus);
    uint16_t* const wf = static_cast<uint16_t*>(w1p);
    uint16_t* const wp = wf + (size_t)dh * kLgDl;
    hipLaunchKernelGGL(w1_pieces_kernel, dim3(dh / 8 * kLgDl / 256), dim3(256), 0, stream, (const uint16_t*)w1, dh, wf, wp);
    if (dh == kLgPass)
        hipLaunchKernelGGL(latent_grad_kernel<1>, dim3(parts), dim3(kLgThreads), 0, stream, dhs, (const uint16_t*)latents, wf, wp,
                           uniq, n_unique, max_u, (uint16_t*)dlat, part);
    else
        hipLaunchKernelGGL(latent_grad_kernel<2>, dim3(parts), dim3(kLgThreads), 0, stream, dhs, (const uint16_t*)latents, wf, wp,
                           uniq, n_unique, max_u, (uint16_t*)dlat, part);
    return launch_gemm_reduce(part, parts, dh, kLgDl, 1.0f, true, dw1, kLgDl, stream);
}

}  // namespace ethos
