// Interface between the GEMM dispatch and the register-staged tiles (gemm_staged.hip).
#pragma once
#include "common.h"

namespace axhip {

struct StagedArgs {
    const void *A, *B;                          // fp32 A; B fp32, or int8 [N, K]
    float *C;
    int64_t M, N, K, lda, ldb, ldc;
    int64_t stride_a, stride_b, stride_c;       // elements between batch members
    int64_t k_range, stride_z;                  // K per range (a multiple of 64, or all of K) and elements between the ranges' outputs
    float alpha, beta;
    const float *col_scale, *bias;
    int act;
};

// The register-staged tiles: any alignment, any K from 32 (fp32) or 64 (int8 weights) up; g.k_range is set to K by the caller
// and cut into ranges here where that pays.  -1: not taken (smaller K, row pitches of 4 Mi elements and more).
// may_split: K may be cut into ranges, whose sums meet in the shared workspace.  Only for a single product, and only for callers
// that keep nothing there: attention's score matrix and the partial sums of an outer K split are operands and results there.
int staged_f32(const StagedArgs &g, int transa, int transb, int64_t batch, bool may_split);
// The same products in bf16 terms on the bf16 matrix core, at fp32 accuracy.
int split_f32(const StagedArgs &g, int transa, int transb, int64_t batch, bool may_split);
// What split_f32 would choose for a single product whose K may be cut into ranges, and the time that it reckons with.
struct StagedChoice {
    bool is_128x128;
    int64_t ranges;
    float us;
};
StagedChoice split_choice(const StagedArgs &g);
// Whether split_f32 would form this batch on its 128x128 tiles.
bool split_is_128x128(const StagedArgs &g, int64_t batch);
int staged_i8w(const StagedArgs &g);
// What a product cut into ranges of K reports when they were formed in bf16 terms (fp32 ranges: sgemm_splitk).
constexpr const char *kSplitTermsName = "sgemm_splitk_x3";
// Batches of A * B^T with K = 32, 64, 96 or 128 in bf16 terms, B held in registers (gemm_nt_terms.hip).  -1: not taken.
int nt_terms(const StagedArgs &g, int64_t batch);
// Batches of A * B with N up to 32 or 65..128 in bf16 terms, a wave over all columns (gemm_nn_terms.hip).  -1: not taken.
int nn_terms(const StagedArgs &g, int64_t batch);

// Adds `splits` partial products [M, N] in order and applies alpha, beta, bias and activation (gemm_f32.hip).
int splitk_finish(const float *part, int64_t splits, int64_t M, int64_t N, float alpha, float beta, const float *bias, int act,
                  float *C, int64_t ldc);

}  // namespace axhip
