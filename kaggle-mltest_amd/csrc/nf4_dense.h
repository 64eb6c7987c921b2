// The 16-bit GEMM behind the large products: the weight dequantized once into a workspace, then
// multiplied by a kernel that only stages and multiplies (nf4_dense.hip).
#pragma once

#include "nf4_common.h"

// One LoRA term: out[m, p] += scale * sum_j l(p, j) t[m, j] for p_lo <= p < p_hi.
struct DenseSlab {
    const uint16_t *l;      // element (p, j) at l[(p - p_lo) * lp + j * lr]
    const uint16_t *t;      // [M, rank]
    int64_t lp, lr;
    int64_t p_lo, p_hi;
    float scale;
    int rank;
    int vec_l, vec_t;       // 16-byte loads of 8 consecutive j allowed
};

// out[m, p] = sum_r w[p, r] act[m, r] (+ LoRA terms) (+ bias[p]), r contiguous in both operands.
struct DenseArgs {
    // w in strips of 128 rows p (the last one's missing rows are never read into a stored
    // output): per 64 reduction values a 16 KB block, row r at 128 r, 8-value chunk c of it at c ^ ((r >> 1) & 7)
    const uint16_t *w;
    const uint16_t *act;    // [M, R], row stride ld_act (a multiple of 8), 16-byte aligned
    int64_t ld_act;
    int64_t P, M, R;        // R a multiple of 64
    uint16_t *out;
    int64_t ld_out;         // multiple of 8, out 16-byte aligned
    const uint16_t *bias;   // [P] or null
    int nslab;
    DenseSlab slab[NF4_MAX_SEGMENTS];
    // the tiling (DensePlan)
    int64_t blocks0, per_split, p_tail;
    int splits;
    float *partial;         // splits > 1: [splits][M][P], to be reduced by the caller
};

// blocks0 workgroups of 256x256 tiles, each tile's reduction over `splits` of them, and
// blocks1 of 128x128 tiles over the rows from p_tail on.
struct DensePlan {
    double cost;            // us, the split's reduction included
    int64_t blocks0, blocks1;
    int64_t per_split, p_tail;
    int splits;
};

DensePlan dense_plan(int64_t P, int64_t M, int64_t R);
int dense_gemm(DenseArgs &a, const DensePlan &p, int dtype, hipStream_t st);

// The stacked weights (one width, a multiple of 128; power-of-two block sizes from 64 on) as the
// strips of DenseArgs::w: P = sum rows, R = cols, or transposed (rows multiples of 64) P = cols,
// R = sum rows.
int dequant_strips(const nf4_weight *ws, int nw, bool transposed, void *out, int dtype, hipStream_t st);
