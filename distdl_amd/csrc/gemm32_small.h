// The fp32 products that linear_f32_small.hip and linear_f32_split.hip compute, and when.
#ifndef DDL_GEMM32_SMALL_H
#define DDL_GEMM32_SMALL_H
#include "gemm_tiles.h"

namespace ddl {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

// Global memory takes the four floats at any alignment: one by one, rows that are no multiple of four went out in four times
// the stores (the partial sums of M 3551, N 6575 135 us instead of 88).
__device__ inline void store_four(float* __restrict__ dst, int64_t n, int64_t N, const floatx4& v) {
    if (n + 3 < N) {
        typedef floatx4 any __attribute__((aligned(4)));
        *reinterpret_cast<any*>(dst) = v;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) dst[e] = v[e];
    }
}

// The bias of columns n .. n + 3 (zeros without one, and past the end).
__device__ inline floatx4 bias_of(const float* __restrict__ bias, int64_t n, int64_t N) {
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float f = bias[n + e < N ? n + e : N - 1];
            b[e] = n + e < N ? f : 0.f;
        }
    }
    return floatx4{b[0], b[1], b[2], b[3]};
}

struct Small32 {
    int groups = 0;           // 0: not taken; 1, 2, 4: tiles of 64 x 64, 32 x 64, 32 x 32
    int edge = 0;             // not 0: linear_f32_split.hip on tiles of edge x edge instead
    double us = 0;            // estimate
    int splits = 1;           // workgroups the reduction of a tile is split over
    int64_t workspace = 0;    // floats for the splits' sums
};

// The cheapest way linear_f32_small.hip has for this product within `workspace` floats; groups 0 if there are too many tiles.
Small32 plan_small32(int64_t M, int64_t N, int64_t K, int cus, int64_t workspace);

// The same for linear_f32_split.hip, next to `other`: `edge` is 0 if that is the cheaper one.
Small32 plan_split32(int64_t M, int64_t N, int64_t K, int cus, int64_t workspace, const Small32& other);

// Launches the product of `part` (its tile counts are set here) as planned; `partial` holds the splits' sums.
int run_small32(const char* who, const Small32& plan, bool xt, bool wt, const PartOf<float>& part, float* partial, int dev, hipStream_t s);

// The adjoint of a linear shard, dx[M, K], dw[N, K] and db[N] from dy[M, N], in one launch (and one that adds split reductions).
struct AdjointPlan32 {
    int groups_x = 0, groups_w = 0;     // tiles, as in Small32; 0: not taken
    int splits_x = 1, splits_w = 1;
    bool first_w = false;
    int64_t workspace = 0;
};
AdjointPlan32 plan_adjoint32(int64_t M, int64_t N, int64_t K, bool want_db, int cus, int64_t workspace, const Small32& x, const Small32& w);

// `dx` and `dw` describe the products dy . w and dy^T . x, `db` may be null.
int run_adjoint32(const AdjointPlan32& plan, const PartOf<float>& dx, const PartOf<float>& dw, float* db, float* workspace, hipStream_t s);

int run_split32(const Small32& plan, bool xt, bool wt, const PartOf<float>& part, float* partial, hipStream_t s);

// Adds the splits' sums and the bias: `partial` holds, split by split and tile by tile, blocks x blocks (2 or 4) blocks of
// 32 x 32, m first, each in the order of the matrix instruction's result.
int sum_small32(const PartOf<float>& part, int blocks, int splits, const float* partial, hipStream_t s);

}  // namespace ddl
#endif  // DDL_GEMM32_SMALL_H
