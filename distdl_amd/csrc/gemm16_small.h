// The 16-bit products that linear_small.hip and linear_any.hip compute, and when.
#ifndef DDL_GEMM16_SMALL_H
#define DDL_GEMM16_SMALL_H
#include "gemm16_elements.h"

namespace ddl {

typedef PartOf<uint16_t> Part16;

struct Small16 {
    enum Kind { kNone, kSkinny, kTiles, kAny, kThin };
    Kind kind = kNone;
    int groups = 1;              // kTiles: groups of wavefronts of a workgroup the reduction is split over (1 or 2)
    int edge = 1;                // kAny: tiles of 64 (1) or 128 (2) rows and columns
    int splits = 1;              // kTiles, kAny: workgroups the reduction of a tile is split over
    int64_t workspace = 0;       // floats for the splits' sums
    double us = 0;               // estimate, if taken
};

// The cheapest way linear_small.hip has for this product within `workspace` floats, kNone if that is not below
// `large_us`, the estimate for the large tiles (microseconds).
Small16 plan_small16(bool xt, bool wt, int64_t M, int64_t N, int64_t K, int cus, int64_t workspace, double large_us);

// The same of linear_any.hip for operands that are not aligned to 16 bytes (kAny, kThin or kNone): against `large_us` and
// copying both operands.
Small16 plan_any16(bool xt, bool wt, int64_t M, int64_t N, int64_t K, int cus, int64_t workspace, double large_us);

// Launches the product of `part` (its tile counts are set here) as planned; `partial` holds the splits' sums.
int run_small16(const char* who, const Small16& plan, bool f16, bool xt, bool wt, const Part16& part, float* partial, int dev, hipStream_t s);
// The adjoint of a linear shard, dx[M, K], dw[N, K] and db[N] from dy[M, N], in one launch (and one that adds split reductions).
struct AdjointPlan16 {
    int edge_x = 0, edge_w = 0;              // tiles of 64 (1) or 128 (2); 0: not taken
    int splits_x = 1, splits_w = 1;
    bool first_w = false;
    int64_t workspace = 0;
};
constexpr int64_t kAdjointRows = 16384;      // of dy, for its column sums

// Against `apart_us`, the estimate for the two products one after the other.
AdjointPlan16 plan_adjoint16(int64_t M, int64_t N, int64_t K, bool aligned, bool want_db, int cus, int64_t workspace, double apart_us);

// `dx` and `dw` describe the products as run_any16 has them (dy . w and dy^T . x), `db` may be null.
int run_adjoint16(const AdjointPlan16& plan, bool f16, const Part16& dx, const Part16& dw, void* db, float* workspace, hipStream_t s);

int run_any16(const Small16& plan, bool f16, bool xt, bool wt, const Part16& part, float* partial, hipStream_t s);

}  // namespace ddl
#endif  // DDL_GEMM16_SMALL_H
