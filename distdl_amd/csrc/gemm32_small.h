// The fp32 products that linear_f32_small.hip computes, and when.
#ifndef DDL_GEMM32_SMALL_H
#define DDL_GEMM32_SMALL_H
#include "gemm_tiles.h"

namespace ddl {

struct Small32 {
    int groups = 0;           // 0: not taken; 1, 2, 4: tiles of 64 x 64, 32 x 64, 32 x 32
    int splits = 1;           // workgroups the reduction of a tile is split over
    int64_t workspace = 0;    // floats for the splits' sums
};

// The cheapest way linear_f32_small.hip has for this product within `workspace` floats; groups 0 if that is not below
// `other_us`, the estimate for the other kernels (microseconds).
Small32 plan_small32(int64_t M, int64_t N, int64_t K, int cus, int64_t workspace, double other_us);

// Launches the product of `part` (its tile counts are set here) as planned; `partial` holds the splits' sums.
int run_small32(const char* who, const Small32& plan, bool xt, bool wt, const PartOf<float>& part, float* partial, int dev, hipStream_t s);

}  // namespace ddl
#endif  // DDL_GEMM32_SMALL_H
