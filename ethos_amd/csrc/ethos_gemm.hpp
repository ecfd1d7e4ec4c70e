// Matrix products of the training path with float32 results (gemm.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace ethos {

// C[m][n] = alpha * sum_k A[m][k] B[k][n] (+ bias[n]), accumulated in float32.  Each operand
// is float32 or bf16 and stored either with k contiguous ([m][k] / [n][k], "K") or with k as
// the row ([k][m] / [k][n], "R").  Sizes: k-contiguous operands need k % 8 == 0 and 16-byte
// aligned rows; row-wise bf16 operands an even column count and 4-byte aligned rows.
struct Gemm {
    const void* a = nullptr;
    const void* b = nullptr;
    void* c = nullptr;
    const void* bias = nullptr;        // [n] of B's type (not with split > 1)
    const int32_t* a_rows = nullptr;   // K-stored A: row m of A is row a_rows[m] of `a`
    int64_t a_limit = INT64_MAX;       // an a_rows entry outside [0, a_limit) is a row of zeros
    const int32_t* b_rows = nullptr;   // R-stored B: row k of B is row b_rows[k] of `b`
    const int32_t* c_rows = nullptr;   // row m of C is row c_rows[m] of `c`
    const int32_t* dyn = nullptr;      // device count: m (or, dyn_k, k) is min(m, *dyn)
    int64_t m = 0, k = 0;
    int n = 0;
    int64_t lda = 0, ldb = 0, ldc = 0;
    float alpha = 1.0f;
    bool dyn_k = false;
    bool out_bf16 = false;             // C is bf16 (rounded to nearest even), else float32
    bool transposed = false;           // C is stored [n][m], ldc its row length
    int epilogue = 0;                  // kGemmPlain, or on the sum (alpha, bias, bf16 unused):
    int split = 1;                     // reduction split over this many workgroups per tile:
    float* part = nullptr;             // [split][m][n] (or [n][m]) float32 partial sums
};

enum GemmEpilogue {
    kGemmPlain,
    kGemmGelu,      // C = gelu(sum)
    kGemmGeluGrad,  // C = gelu'(sum) C, in place
};

enum GemmForm {
    kGemmBK_BK,  // A bf16 K, B bf16 K
    kGemmBK_BR,  // A bf16 K, B bf16 R
    kGemmFK_BK,  // A float32 K, B bf16 K
    kGemmFK_BR,  // A float32 K, B bf16 R
    kGemmFR_BR,  // A float32 R, B bf16 R
    kGemmFK_FK,  // float32 both
    kGemmFK_FR,
    kGemmFR_FR,
};

// Splits of a product of m x n outputs over k so that the chip has about two workgroups per
// CU, each with at least 256 of the reduction.
int gemm_split(int64_t m, int n, int64_t k, int num_cus);
int launch_gemm(GemmForm form, const Gemm& g, int num_cus, hipStream_t stream);
// c = alpha * (the sum of `split` partial results [rows][cols], in order).
int launch_gemm_reduce(const float* part, int split, int64_t rows, int64_t cols, float alpha, bool out_bf16, void* c, int64_t ldc,
                       hipStream_t stream);

// d latents and d W1 of the experts from dh in one pass (latent_grad.hip); w1p: d_hidden x 128
// floats of workspace (W1 in two orders), part: latent_grad_parts() x d_hidden x 128 floats.
// Taken when up to 16,384 unique experts or more are possible (a tile of 64 for each CU: 49 us against 94
// as products); with fewer, part of the CUs would be idle in both forms and the products, which
// spread over more workgroups, are kept.
constexpr int64_t kLatentGradRows = 16384;
bool latent_grad_fits(int64_t max_u, int dl, int dh);
int latent_grad_parts(int64_t max_u, int num_cus);
int launch_latent_grad(const float* dhs, const void* latents, const void* w1, const int32_t* uniq, const int32_t* n_unique,
                       int64_t max_u, int dh, void* w1p, float* part, void* dlat, void* dw1, int num_cus, hipStream_t stream);

}  // namespace ethos
