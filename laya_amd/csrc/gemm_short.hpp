// Products too short for the 128 x 128 and 256-wide tiles of gemm.hip to fill the chip (gemm_short.hip).
#pragma once
#include "common.hpp"

namespace laya {

enum class ShortEpilogue {
    Store,       // C = acc (+ bias) (+ R)
    Accumulate,  // C += acc
    Rope,        // C = rotated acc (+ bias) in the first rope_cols columns (heads of 64), acc (+ bias) in the rest
    Geglu,       // B's rows are [first half; second half]: both halves into C, act = gelu(first)·second
};

struct ShortGemm {
    const float *A, *B, *bias, *R;
    float* C;
    long lda, ldb, ldc, ldr;
    int M, N, K;
    unsigned* amax;  // optional magnitude word group of C (Geglu: of act)
    const int* rope_pos;
    const float *rope_cos, *rope_sin;
    int rope_cols;
    float* act;
    __bf16* act16;
    int inter;
    int tiles_m, tiles_n;  // set by the launchers
};

// Whether the product runs here, under the context's precision for its layout (two-piece fp16 products, or bf16
// operands): its shape allows it and these tiles take less time than `other`, gemm.hip's in microseconds.
bool short_gemm_pays(const laya_ctx* ctx, GemmLayout layout, ShortEpilogue ep, const ShortGemm& g, double other);
void short_gemm(laya_ctx* ctx, GemmLayout layout, ShortEpilogue ep, ShortGemm g);
// A linear layer's dX (NN, Store) and dW (TN, Accumulate) in one launch. lines: fp32 operands scaled by row and column,
// for pairs that exact three-piece splits would compute otherwise.
bool short_pair_pays(const laya_ctx* ctx, const ShortGemm& nn, const ShortGemm& tn, bool lines, double other);
void short_gemm_pair(laya_ctx* ctx, ShortGemm nn, ShortGemm tn, bool lines);

}  // namespace laya
