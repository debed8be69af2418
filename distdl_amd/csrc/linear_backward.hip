// Helpers of the DistributedLinear shard backward (the adjoint of
// torch.nn.functional.linear, reference: nn/linear.py:103, nn/linear_ag.py:486):
//
//   dx[M,K] = dy[M,N] . w[N,K]          reduction over N
//   dw[N,K] = dy[M,N]^T . x[M,K]        reduction over M
//   db[N]   = sum over m of dy[m,N]
//
// ddl_linear_backward runs what is wanted of the three: the products read w, dy
// and x where they lie (ddl_gemm_ws), db is a column sum with fp32 accumulation.
// Large 16-bit products whose operands cannot be read in place are transposed
// into temporaries by the caller (ddl_transpose_2d) and go through ddl_linear.
#include "colsum.h"
#include "gemm16_small.h"
#include "gemm32_small.h"

#include <type_traits>

namespace ddl {
namespace {

constexpr int kTile = 64;      // elements per tile edge
constexpr int kBlock = 256;

__device__ inline void store16(uint16_t* p, uint4 q) {
    struct __attribute__((packed, aligned(2))) Any {
        uint32_t word[4];
    };
    *reinterpret_cast<Any*>(p) = Any{{q.x, q.y, q.z, q.w}};
}

// Elements [first, first + 8) of a row of `n`, zeros past its end.
__device__ inline uint4 load_piece(const uint16_t* row, int64_t first, int64_t n) {
    if (first + 8 <= n) return load16(row + first);
    uint32_t q[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (first + e < n) q[e >> 1] |= static_cast<uint32_t>(row[first + e]) << (16 * (e & 1));
    return make_uint4(q[0], q[1], q[2], q[3]);
}

// dst[c, r] = src[r, c] for 16-bit elements, and zeros in the columns rows .. width of dst.  A 64 x 64 tile goes through
// LDS: rows are read 16 bytes per lane at whatever address they have; a lane reads 8 rows of two source columns back, 4
// bytes each, sorts them apart and writes 16 bytes to each of two rows of dst.  The LDS row pitch of 66 elements (33
// dwords) puts the 64 lanes of a wavefront on 64 banks.  The tiles of an XCD are neighbours, so that the lines which two
// tiles of a row share come from its L2.  Bound by memory: dy [5066, 3572] bf16, whose rows are not 16 bytes apart, into
// a zeroed [3572, 5072] took 52 us by 2-byte accesses, after a clear of 7; now 13.4 for both, at 5.4 TB/s.
__global__ __launch_bounds__(kBlock) void transpose16_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                             int64_t rows, int64_t cols, int64_t ld_src, int64_t ld_dst,
                                                             int64_t width, uint32_t tiles_c, uint32_t tiles, uint32_t per_xcd) {
    __shared__ uint32_t tile[kTile][kTile / 2 + 1];
    const uint32_t b = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (b >= tiles) return;
    const uint32_t tr = b / tiles_c, tc = b - tr * tiles_c;
    const int64_t r0 = static_cast<int64_t>(tr) * kTile, c0 = static_cast<int64_t>(tc) * kTile;
    const int t = threadIdx.x;
    // 8 lanes per row (8 x 8 elements), 32 rows per pass
    uint4 q[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int64_t gr = r0 + (t >> 3) + 32 * p, gc = c0 + (t & 7) * 8;
        q[p] = gr < rows ? load_piece(src + gr * ld_src, gc, cols) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        uint32_t* to = &tile[(t >> 3) + 32 * p][(t & 7) * 4];
        to[0] = q[p].x, to[1] = q[p].y, to[2] = q[p].z, to[3] = q[p].w;
    }
    __syncthreads();
    // 8 lanes per pair of output rows, 8 source rows each
    const int pair = t >> 3, first = (t & 7) * 8;
    uint32_t even[4], odd[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t lo = tile[first + 2 * e][pair], hi = tile[first + 2 * e + 1][pair];
        even[e] = (lo & 0xFFFFu) | (hi << 16);
        odd[e] = (lo >> 16) | (hi & 0xFFFF0000u);
    }
    const int64_t gc = c0 + 2 * pair, gr = r0 + first;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (gc + h >= cols) break;
        const uint32_t* v = h ? odd : even;
        uint16_t* d = dst + (gc + h) * ld_dst + gr;
        if (gr + 8 <= width) {
            store16(d, make_uint4(v[0], v[1], v[2], v[3]));
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (gr + e < width) d[e] = static_cast<uint16_t>(v[e >> 1] >> (16 * (e & 1)));
        }
    }
}

// dst[r, c] = src[r, c], and zeros in the columns cols .. 8 * pieces of dst, whose rows lie end to end: 16 bytes a lane.
// [5066, 3572] bf16 in 16.7 us; a clear and a box copy took 25.
constexpr int kPadPieces = 4;   // per lane

__global__ __launch_bounds__(kBlock) void pad16_kernel(const uint16_t* __restrict__ src, uint4* __restrict__ dst, uint32_t total,
                                                       uint32_t pieces, int64_t cols, int64_t ld_src) {
    const uint32_t first = blockIdx.x * (kBlock * kPadPieces) + threadIdx.x;
    uint4 q[kPadPieces];
#pragma unroll
    for (int p = 0; p < kPadPieces; ++p) {
        const uint32_t i = first + p * kBlock < total ? first + p * kBlock : total - 1;
        const uint32_t r = i / pieces;
        q[p] = load_piece(src + static_cast<int64_t>(r) * ld_src, static_cast<int64_t>(i - r * pieces) * 8, cols);
    }
#pragma unroll
    for (int p = 0; p < kPadPieces; ++p)
        if (first + p * kBlock < total) dst[first + p * kBlock] = q[p];
}

// Stage 1 of the column sum: workgroup (strip, split) adds rows
// [split * rows_per_split, ...) of a 64-column strip in fp32 and writes 64
// partial sums to partial[split, col].  8 lanes cover the 64 columns of a row,
// 32 rows are in flight per pass; LDS folds the 32 row groups.
template <int DT>
__global__ __launch_bounds__(kBlock) void colsum_partial_kernel(const typename Elem<DT>::type* __restrict__ a, int64_t rows, int64_t cols,
                                                                int64_t ld, int64_t rows_per_split, float* __restrict__ partial,
                                                                int strips) {
    __shared__ float fold[32][kTile + 1];
    const int split = blockIdx.x / strips, strip = blockIdx.x - split * strips;
    const int t = threadIdx.x;
    const int g = t >> 3, c = (t & 7) * 8;
    const int64_t gc = static_cast<int64_t>(strip) * kTile + c;
    const int64_t r_begin = split * rows_per_split;
    const int64_t r_end = r_begin + rows_per_split < rows ? r_begin + rows_per_split : rows;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (gc + 8 <= cols) {
        for (int64_t r = r_begin + g; r < r_end; r += 32) {
            float v[8];
            Elem<DT>::load8(a + r * ld + gc, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += v[e];
        }
    } else {
        for (int64_t r = r_begin + g; r < r_end; r += 32) {
            const typename Elem<DT>::type* s = a + r * ld + gc;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (gc + e < cols) acc[e] += Elem<DT>::load(s + e);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) fold[g][c + e] = acc[e];
    __syncthreads();
    if (t < kTile) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 32; ++k) s += fold[k][t];
        const int64_t col = static_cast<int64_t>(strip) * kTile + t;
        if (col < cols) partial[static_cast<int64_t>(split) * cols + col] = s;
    }
}

// Stage 2: out[col] = sum over splits of partial[split, col], rounded to the element type.  A workgroup
// per 64-column strip; lane group t / 64 adds every fourth split (eight
// independent loads in flight), LDS folds the four groups.
template <int DT>
__global__ __launch_bounds__(kBlock) void colsum_final_kernel(const float* __restrict__ partial, int64_t cols, int splits,
                                                              typename Elem<DT>::type* __restrict__ out) {
    constexpr int kGroups = kBlock / kTile;
    __shared__ float fold[kGroups][kTile];
    const int g = threadIdx.x / kTile, t = threadIdx.x % kTile;
    const int64_t col = static_cast<int64_t>(blockIdx.x) * kTile + t;
    float s = 0.f;
    if (col < cols) {
        int k = g;
        for (; k + 7 * kGroups < splits; k += 8 * kGroups) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = partial[static_cast<int64_t>(k + u * kGroups) * cols + col];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
        for (; k < splits; k += kGroups) s += partial[static_cast<int64_t>(k) * cols + col];
    }
    fold[g][t] = s;
    __syncthreads();
    if (g == 0 && col < cols) {
        float r = 0.f;
#pragma unroll
        for (int k = 0; k < kGroups; ++k) r += fold[k][t];
        Elem<DT>::store(out + col, r);
    }
}

// The column sum of few rows in one launch, see colsum.h.
constexpr int kOneBlock = 1024;

template <int DT>
__global__ __launch_bounds__(kOneBlock) void colsum_one_kernel(const typename Elem<DT>::type* __restrict__ a, int64_t rows, int64_t cols,
                                                               int64_t ld, typename Elem<DT>::type* __restrict__ out) {
    __shared__ char lds[colsum_lds_bytes(DT, kOneBlock)];
    colsum_strip<DT, kOneBlock, 1>(a, rows, cols, ld, out, blockIdx.x, gridDim.x, lds);
}

}  // namespace
}  // namespace ddl

extern "C" int ddl_transpose_2d(const void* src, void* dst, int64_t rows, int64_t cols, int64_t ld_src, int64_t ld_dst,
                                int elem_size, void* stream) {
    return ddl_transpose_padded(src, dst, rows, cols, ld_src, ld_dst, rows, elem_size, stream);
}

extern "C" int ddl_transpose_padded(const void* src, void* dst, int64_t rows, int64_t cols, int64_t ld_src, int64_t ld_dst,
                                    int64_t width, int elem_size, void* stream) {
    using namespace ddl;
    if (rows < 0 || cols < 0 || ld_src < cols || width < rows || ld_dst < width)
        return fail(DDL_E_ARG, "transpose: rows=%lld cols=%lld ld_src=%lld ld_dst=%lld", (long long)rows, (long long)cols,
                    (long long)ld_src, (long long)ld_dst);
    if (elem_size != 2) return fail(DDL_E_UNSUPP, "transpose: element size %d (only 2-byte elements)", elem_size);
    if (width == 0 || cols == 0) return 0;
    if ((!src && rows > 0) || !dst) return fail(DDL_E_ARG, "transpose: null pointer");
    if (!aligned_to(src, 2) || !aligned_to(dst, 2)) return fail(DDL_E_ALIGN, "transpose: pointer misaligned");
    const int64_t tiles_r = (width + kTile - 1) / kTile, tiles_c = (cols + kTile - 1) / kTile;
    if (tiles_c > 0x7FFFFF00ll || tiles_r > 0x7FFFFF00ll / tiles_c) return fail(DDL_E_UNSUPP, "transpose: too many tiles");
    const uint32_t tiles = static_cast<uint32_t>(tiles_r * tiles_c), per_xcd = (tiles + kXcds - 1) / kXcds;
    hipLaunchKernelGGL(transpose16_kernel, dim3(per_xcd * kXcds), dim3(kBlock), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), rows, cols, ld_src, ld_dst, width,
                       static_cast<uint32_t>(tiles_c), tiles, per_xcd);
    return check_launch("transpose16_kernel");
}

extern "C" int ddl_pad_rows(const void* src, void* dst, int64_t rows, int64_t cols, int64_t ld_src, int64_t width, int elem_size,
                            void* stream) {
    using namespace ddl;
    if (rows < 0 || cols < 0 || ld_src < 0 || width < cols || width % 8 != 0)
        return fail(DDL_E_ARG, "pad: rows=%lld cols=%lld ld_src=%lld width=%lld", (long long)rows, (long long)cols, (long long)ld_src,
                    (long long)width);
    if (elem_size != 2) return fail(DDL_E_UNSUPP, "pad: element size %d (only 2-byte elements)", elem_size);
    if (rows == 0 || width == 0) return 0;
    if ((!src && cols > 0) || !dst) return fail(DDL_E_ARG, "pad: null pointer");
    if (!aligned_to(src, 2) || !aligned_to(dst, 16)) return fail(DDL_E_ALIGN, "pad: pointer misaligned");
    // Lanes number the pieces in 32 bits: slabs of rows that they reach, and no row is longer than that.
    const int64_t pieces = width / 8, most = 0x7FFF0000ll / pieces;
    if (most < 1) return fail(DDL_E_UNSUPP, "pad: rows of %lld elements", (long long)width);
    for (int64_t r = 0; r < rows; r += most) {
        const uint32_t total = static_cast<uint32_t>((rows - r < most ? rows - r : most) * pieces);
        hipLaunchKernelGGL(pad16_kernel, dim3((total + kBlock * kPadPieces - 1) / (kBlock * kPadPieces)), dim3(kBlock), 0,
                           static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(src) + r * ld_src,
                           static_cast<uint4*>(dst) + r * pieces, total, static_cast<uint32_t>(pieces), cols, ld_src);
        if (int rc = check_launch("pad16_kernel")) return rc;
    }
    return 0;
}

namespace ddl {

// Up to 128 KiB per workgroup of 16 columns: about 4 us on one CU; and fewer than the 2^32 threads a launch may have.
bool colsum_in_one_launch(int64_t rows, int64_t cols, int64_t elem_size) {
    return rows <= 131072 / (kNarrow * elem_size) && (cols + kNarrow - 1) / kNarrow <= 0xFFFFFFFFll / kOneBlock;
}

}  // namespace ddl

namespace ddl {
namespace {

template <int DT>
int run_colsum(const void* a, int64_t rows, int64_t cols, int64_t ld, void* out, float* workspace, int64_t splits,
               int64_t rows_per_split, int64_t strips, hipStream_t s) {
    typedef typename Elem<DT>::type T;
    if (colsum_in_one_launch(rows, cols, sizeof(T))) {
        const dim3 grid(static_cast<uint32_t>((cols + kNarrow - 1) / kNarrow));
        hipLaunchKernelGGL((colsum_one_kernel<DT>), grid, dim3(kOneBlock), 0, s, static_cast<const T*>(a), rows, cols, ld, static_cast<T*>(out));
        return check_launch("colsum_one_kernel");
    }
    hipLaunchKernelGGL((colsum_partial_kernel<DT>), dim3(static_cast<uint32_t>(strips * splits)), dim3(kBlock), 0, s,
                       static_cast<const T*>(a), rows, cols, ld, rows_per_split, workspace, static_cast<int>(strips));
    const int rc = check_launch("colsum_partial_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL((colsum_final_kernel<DT>), dim3(static_cast<uint32_t>(strips)), dim3(kBlock), 0, s, workspace, cols,
                       static_cast<int>(splits), static_cast<T*>(out));
    return check_launch("colsum_final_kernel");
}

}  // namespace
}  // namespace ddl

extern "C" int ddl_colsum(const void* a, int dtype, int64_t rows, int64_t cols, int64_t ld, void* out, float* workspace,
                          int64_t workspace_elems, void* stream) {
    using namespace ddl;
    if (dtype != DDL_DT_BF16 && dtype != DDL_DT_F16 && dtype != DDL_DT_F32) return fail(DDL_E_UNSUPP, "colsum: dtype %d (bf16, f16 and f32 only)", dtype);
    if (rows < 0 || cols < 0 || ld < cols) return fail(DDL_E_ARG, "colsum: rows=%lld cols=%lld ld=%lld", (long long)rows, (long long)cols, (long long)ld);
    if (cols == 0) return 0;
    const int es = dtype == DDL_DT_F32 ? 4 : 2;
    const bool one_launch = colsum_in_one_launch(rows, cols, es);
    if (!out || (!workspace && !one_launch) || (rows > 0 && !a)) return fail(DDL_E_ARG, "colsum: null pointer");
    if (!aligned_to(a, es) || !aligned_to(out, es) || !aligned_to(workspace, 4)) return fail(DDL_E_ALIGN, "colsum: pointer misaligned");
    // as many row splits as the workspace holds, up to 64 and to 128 rows per split
    int64_t splits = one_launch ? 1 : workspace_elems / cols;
    if (splits < 1) return fail(DDL_E_ARG, "colsum: workspace of %lld floats is smaller than one row of %lld", (long long)workspace_elems, (long long)cols);
    if (splits > 64) splits = 64;
    const int64_t by_rows = (rows + 127) / 128;
    if (splits > by_rows) splits = by_rows > 0 ? by_rows : 1;
    const int64_t rows_per_split = rows > 0 ? (rows + splits - 1) / splits : 1;
    const int64_t strips = (cols + kTile - 1) / kTile;
    if (strips * splits > 0x7FFFFFFFll) return fail(DDL_E_UNSUPP, "colsum: too many workgroups");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == DDL_DT_BF16) return run_colsum<0>(a, rows, cols, ld, out, workspace, splits, rows_per_split, strips, s);
    if (dtype == DDL_DT_F16) return run_colsum<1>(a, rows, cols, ld, out, workspace, splits, rows_per_split, strips, s);
    return run_colsum<2>(a, rows, cols, ld, out, workspace, splits, rows_per_split, strips, s);
}

namespace ddl {

AdjointPlan16 adjoint16(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t lddy, bool aligned, bool want_db, int64_t workspace);
Small32 plan32(int64_t a_rs, int64_t a_ks, int64_t b_rs, int64_t b_ks, int64_t M, int64_t N, int64_t K, int cus, int64_t workspace);

constexpr int64_t kAdjointRows32 = 2048;   // longer column sums stay in two stages, whose partial sums are shorter

// The same in fp32: where both products go to linear_f32_small.hip.
static AdjointPlan32 adjoint32(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t lddy, bool want_db, int64_t workspace) {
    int dev = 0;
    const int cus = compute_units(dev);
    // strides of 1 and 1 say nothing about the order of an operand
    if (M < 2 || N < 2 || K < 2 || ldx < 2 || ldw < 2 || lddy < 2) return AdjointPlan32{};
    const Small32 x = plan32(lddy, 1, 1, ldw, M, K, N, cus, INT64_MAX), w = plan32(1, lddy, 1, ldx, N, K, M, cus, INT64_MAX);
    return plan_adjoint32(M, N, K, want_db, cus, workspace, x, w);
}

// dx, dw and, `inside`, db in one launch, if that is how they are computed.
struct OneLaunch {
    bool taken = false, inside = false;
    AdjointPlan32 wide;
    AdjointPlan16 narrow;
};

static OneLaunch one_launch(int dtype, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t lddy, bool aligned, bool want_db, int64_t workspace) {
    OneLaunch plan;
    if (dtype == DDL_DT_F32) {
        plan.inside = want_db && M <= kAdjointRows32;
        plan.wide = adjoint32(M, N, K, ldx, ldw, lddy, plan.inside, workspace);
        plan.taken = plan.wide.groups_x != 0;
    } else if (dtype == DDL_DT_BF16 || dtype == DDL_DT_F16) {
        plan.inside = want_db && M <= kAdjointRows;
        plan.narrow = adjoint16(M, N, K, ldx, ldw, lddy, aligned, plan.inside, workspace);
        plan.taken = plan.narrow.edge_x != 0;
    }
    return plan;
}

}  // namespace ddl

extern "C" int ddl_linear_backward_plan(int dtype, int aligned, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t lddy, int want_db,
                                        int64_t workspace_elems, int* plan) {
    using namespace ddl;
    if (M < 1 || N < 1 || K < 1 || !plan) return 0;
    const OneLaunch one = one_launch(dtype, M, N, K, ldx, ldw, lddy, aligned != 0, want_db != 0, workspace_elems);
    if (!one.taken) return 0;
    const bool wide = dtype == DDL_DT_F32;
    plan[0] = wide ? one.wide.groups_x : one.narrow.edge_x, plan[1] = wide ? one.wide.groups_w : one.narrow.edge_w;
    plan[2] = wide ? one.wide.splits_x : one.narrow.splits_x, plan[3] = wide ? one.wide.splits_w : one.narrow.splits_w;
    plan[4] = one.inside;
    return 1;
}

extern "C" int64_t ddl_linear_backward_workspace_at(int dtype, int aligned, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw,
                                                    int64_t lddy, int want_dx, int want_dw, int want_db) {
    // The products and the column sum run one after the other, so they share the workspace.  If not all operands are
    // aligned, a product may still have two that are.
    int64_t most = 0;
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    auto take = [&](int64_t elems) { most = elems > most ? elems : most; };
    if (want_dx && want_dw) {   // both in one launch, with a part of the workspace each
        const ddl::OneLaunch plan = ddl::one_launch(dtype, M, N, K, ldx, ldw, lddy, aligned != 0, want_db != 0, INT64_MAX);
        if (plan.taken) {
            take(plan.wide.workspace + plan.narrow.workspace);
            want_dx = want_dw = 0;
            if (plan.inside) want_db = 0;
        }
    }
    for (int both = aligned ? 1 : 0; both < 2; ++both) {
        if (want_dx) take(ddl_gemm_workspace_at(dtype, both, lddy, 1, 1, ldw, M, K, N));
        if (want_dw) take(ddl_gemm_workspace_at(dtype, both, 1, lddy, 1, ldx, N, K, M));
    }
    if (want_db && !ddl::colsum_in_one_launch(M, N, dtype == DDL_DT_F32 ? 4 : 2)) {
        const int64_t splits = (M + 127) / 128;
        take((splits < 64 ? splits : 64) * N);
    }
    return most;
}

extern "C" int64_t ddl_linear_backward_workspace(int dtype, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t lddy,
                                                 int want_dx, int want_dw, int want_db) {
    return ddl_linear_backward_workspace_at(dtype, 1, M, N, K, ldx, ldw, lddy, want_dx, want_dw, want_db);
}

extern "C" int ddl_linear_backward(const void* x, const void* w, const void* dy, void* dx, void* dw, void* db, int dtype, int64_t M, int64_t N,
                                   int64_t K, int64_t ldx, int64_t ldw, int64_t lddy, float* workspace, int64_t workspace_elems, void* stream) {
    using namespace ddl;
    if (M < 1 || N < 1 || K < 1) return fail(DDL_E_ARG, "linear backward: M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
    if (!dy || (dx && !w) || (dw && !x)) return fail(DDL_E_ARG, "linear backward: null pointer");
    const int es = dtype == DDL_DT_F32 ? 4 : 2;
    if (dx && dw && aligned_to(x, es) && aligned_to(w, es) && aligned_to(dy, es) && aligned_to(dx, es) && aligned_to(dw, es) && aligned_to(db, es) &&
        (!workspace || aligned_to(workspace, 16))) {
        const bool aligned = aligned_to(x, 16) && aligned_to(w, 16) && aligned_to(dy, 16);
        const OneLaunch plan = one_launch(dtype, M, N, K, ldx, ldw, lddy, aligned, db != nullptr, workspace ? workspace_elems : 0);
        if (plan.taken) {
            auto run = [&](auto* element, auto&& launch) {
                using T = std::remove_pointer_t<decltype(element)>;
                PartOf<T> to_x{}, to_w{};
                to_x.x = static_cast<const T*>(dy), to_x.ldx = lddy, to_x.w = static_cast<const T*>(w), to_x.ldw = ldw;
                to_x.y = static_cast<T*>(dx), to_x.ldy = K, to_x.M = M, to_x.N = K, to_x.K = N;
                to_w.x = static_cast<const T*>(dy), to_w.ldx = lddy, to_w.w = static_cast<const T*>(x), to_w.ldw = ldx;
                to_w.y = static_cast<T*>(dw), to_w.ldy = K, to_w.M = N, to_w.N = K, to_w.K = M;
                return launch(to_x, to_w, plan.inside ? db : nullptr);
            };
            const hipStream_t s = static_cast<hipStream_t>(stream);
            const int rc = dtype == DDL_DT_F32
                               ? run(static_cast<float*>(nullptr), [&](auto& to_x, auto& to_w, void* sums) { return run_adjoint32(plan.wide, to_x, to_w, static_cast<float*>(sums), workspace, s); })
                               : run(static_cast<uint16_t*>(nullptr), [&](auto& to_x, auto& to_w, void* sums) { return run_adjoint16(plan.narrow, dtype == DDL_DT_F16, to_x, to_w, sums, workspace, s); });
            return rc || plan.inside || !db ? rc : ddl_colsum(dy, dtype, M, N, lddy, db, workspace, workspace_elems, stream);
        }
    }
    // dx[m, j] = sum_n dy[m, n] w[n, j]: rows of the second operand are the columns of w
    if (dx)
        if (int rc = ddl_gemm_ws(dy, lddy, 1, w, 1, ldw, nullptr, dx, dtype, K, M, K, N, workspace, workspace_elems, stream)) return rc;
    // dw[i, j] = sum_m dy[m, i] x[m, j]: both operands are read down their columns
    if (dw)
        if (int rc = ddl_gemm_ws(dy, 1, lddy, x, 1, ldx, nullptr, dw, dtype, K, N, K, M, workspace, workspace_elems, stream)) return rc;
    if (db) return ddl_colsum(dy, dtype, M, N, lddy, db, workspace, workspace_elems, stream);
    return 0;
}

extern "C" int ddl_colsum_bf16(const void* a, int64_t rows, int64_t cols, int64_t ld, void* out, float* workspace,
                               int64_t workspace_elems, void* stream) {
    return ddl_colsum(a, DDL_DT_BF16, rows, cols, ld, out, workspace, workspace_elems, stream);
}
