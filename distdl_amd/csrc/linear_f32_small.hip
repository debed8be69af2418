// fp32 linear products too small to fill the chip with the 128 x 128 tiles of
// linear_f32_split.hip: y[M,N] = a[M,K] . b[N,K]^T + bias[N] on v_mfma_f32_32x32x2_f32.
//
// Bound by the matrix cores of the CUs that have work (a 64 x 64 tile of K 1024 is
// 14 us on one CU), so tiles are small and the reduction is split wherever that
// gives more CUs a share.  A workgroup is four wavefronts with 32 x 32 of the result
// each: 2 x 2 of them (tile 64 x 64), 1 x 2 in two groups that take alternate k-tiles
// (32 x 64), or one in four groups (32 x 32); the groups' sums meet in LDS.
// `splits` workgroups share the reduction of a tile through a workspace;
// gemm32_small_sum adds their sums in the order of the splits.
//
// A wavefront multiplies one half of a k-tile while the other half, or the first half of the next k-tile, comes
// from LDS, and the requests go out one or two per matrix instruction: where a CU has one workgroup, nothing else
// fills these waits.  All reads of a k-tile first, then its products: a round 0.78 us in two groups and 0.68 in
// one, here 0.57 and 0.54, of which the matrix cores take 0.43 (M 777, N 333, K 1024 17.0 -> 13.0 us, its adjoint
// 22.0 -> 19.4; M = N = K = 1024 26.0 -> 20.9; M 399, N 1115, K 3264 1.5 times as fast; 4000 products of up to 8e9
// operations 1.09 times, their adjoints 1.04).  The last rounds, with decisions in them, have a loop of their own:
// with those in the only loop M 777 took 14.9.
//
// Tiles go from global memory straight into LDS through a ring of stages: k-tiles of
// 32 floats; an operand contiguous along k in rows of 128 bytes whose 16-byte chunks are
// XOR-ed with (row >> 1) & 7 (lane (r = lane % 32, h = lane / 32) reads chunk 2 g + h of row
// r and feeds its four floats to the four matrix instructions of k-group g: any
// assignment of k to lanes and steps is valid if both operands use the same one); an
// operand contiguous along its rows as it lies in memory, in panels of 32 rows x 32
// k-lines of 128 bytes (lane (r, h) reads element r of k-line 8 g + 4 h + e; lines k and
// k + 4 would start on the same bank, so the lines 4..7 of every eight are stored with
// neighbours swapped).  A
// request reads 16 bytes per lane from any 4-byte-aligned address, so pitches and
// lengths are free: only the k-tile that straddles K, and the last one of an operand
// read along rows whose number is no multiple of four (a chunk there runs over into
// the next k-line, which the last one has not), go through registers element by
// element.  (The addresses there are selected, not branched on: with branches the
// compiler kept 360 registers, one workgroup fit on a CU, and the kernel took 1.4 times
// as long.)
//
// linear32_adjoint is dx, dw and db of a linear shard in one launch, for products whose
// workgroups are all resident at once: alone each of the three leaves CUs idle and waits
// for the one before.  M 777, N 333, K 1024 28.1 -> 19.4 us, M 97, N 77, K 603 10.9 -> 5.3, M 108, N
// 192, K 5376 15.8 -> 10.5, M = N = K = 1024 53.9 -> 38.5.  With more workgroups the products fill
// the chip one after the other, and the one launch is slower (M 2078, N 6152, K 276 162, here 243).
#include "colsum.h"
#include "gemm_tiles.h"
#include "gemm32_small.h"
#include <type_traits>

namespace ddl {
namespace {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

constexpr int BK = kRowBytes / 4;   // floats of a k-tile
typedef PartOf<float> Part32;

// Workgroup `number` of the tiles_m x tiles_n x splits of a product.
template <bool XT, bool WT, int NWM, int NWN, int KG, int STAGES>
__device__ __forceinline__ void small_product(const Part32& p, int number, int splits, float* __restrict__ partial, char* lds) {
    constexpr int NW = NWM * NWN, BM = 32 * NWM, BN = 32 * NWN;
    static_assert(NW * KG == 4, "four wavefronts per workgroup");
    constexpr int JW_W = BN / 8 / NW, JW_X = BM / 8 / NW;   // request instructions (1 KiB each) per wavefront and tile
    constexpr int kStage = (BM + BN) * kRowBytes, kX = BN * kRowBytes;   // a stage holds the w tile and then the x tile
    const int ntiles = p.tiles_m * p.tiles_n;
    const int split = number / ntiles, tile = number - split * ntiles;
    int tm, tn;
    tile_of_workgroup(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int64_t M = p.M, N = p.N, K = p.K;
    const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
    const int lane = threadIdx.x & 63, group = __builtin_amdgcn_readfirstlane(threadIdx.x / (NW * 64));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) - group * NW;   // inside its group
    const int l32 = lane & 31, kh = lane >> 5;
    const int sub_w = wave / NWM, sub_x = wave % NWM;   // 32-row block of this wavefront in the w and x tiles

    const int ktiles = static_cast<int>((K + BK - 1) / BK);
    // Tiles from here on go through registers (see the head of the file).
    const bool w_over = WT && N % 4 != 0, x_over = XT && M % 4 != 0;
    const int full_tiles = static_cast<int>((w_over || x_over ? K - 1 : K) / BK);
    const int per = (ktiles + splits - 1) / splits;
    const int t_begin = split * per < ktiles ? split * per : ktiles, t_end = t_begin + per < ktiles ? t_begin + per : ktiles;
    char* const ring = lds + group * (STAGES * kStage);

    // Piece i = NW j + wave of a tile.  Along k: rows 8 i .. + 7, lane l on row l / 8, physical chunk l % 8.  Along rows:
    // panel i / 4, k-lines 8 (i % 4) .. + 7 with neighbours swapped in lines 4 .. 7, rows 4 (l % 8) .. + 3 of the panel.
    // Rows past the end repeat the last one, chunks that start past it the first of the tile; never stored.
    const char* const base_w = reinterpret_cast<const char*>(WT ? p.w + n0 : p.w + n0 * p.ldw);
    const char* const base_x = reinterpret_cast<const char*>(XT ? p.x + m0 : p.x + m0 * p.ldx);
    const u32x4 buf_w = raw_buffer(base_w), buf_x = raw_buffer(base_x);
    const int step_w = WT ? static_cast<int>(p.ldw) * (BK * 4) : BK * 4;
    const int step_x = XT ? static_cast<int>(p.ldx) * (BK * 4) : BK * 4;
    auto chunk_k = [&](bool transposed, int i) {   // first k of this lane's chunk, or its k-line, inside a k-tile
        const int row = i * 8 + (lane >> 3), q = lane >> 3;
        return transposed ? 8 * (i & 3) + (q ^ ((q >> 2) & 1)) : ((lane & 7) ^ ((row >> 1) & 7)) * 4;
    };
    auto chunk_row = [&](bool transposed, int i, int64_t origin, int64_t rows) -> int {   // (first) row inside the tile
        if (!transposed) {
            const int row = i * 8 + (lane >> 3);
            return origin + row < rows ? row : static_cast<int>(rows - 1 - origin);
        }
        const int col = (i >> 2) * 32 + (lane & 7) * 4;
        return origin + col < rows ? col : 0;
    };
    auto lane_offset = [&](bool transposed, int i, int64_t origin, int64_t rows, int64_t ld) -> int {
        const int64_t k = chunk_k(transposed, i), r = chunk_row(transposed, i, origin, rows);
        return static_cast<int>((transposed ? k * ld + r : r * ld + k) * 4);
    };
    int off_w[JW_W], off_x[JW_X];
#pragma unroll
    for (int j = 0; j < JW_W; ++j) off_w[j] = lane_offset(WT, NW * j + wave, n0, N, p.ldw);
#pragma unroll
    for (int j = 0; j < JW_X; ++j) off_x[j] = lane_offset(XT, NW * j + wave, m0, M, p.ldx);
    // One chunk through registers: elements past K or past the rows are zeros.
    auto careful = [&](bool transposed, const char* base, int off, int64_t step, int t, int i, int64_t origin, int64_t rows, char* dst) {
        const int64_t at = off + t * step;
        const int64_t k = static_cast<int64_t>(t) * BK + chunk_k(transposed, i), r = origin + chunk_row(transposed, i, origin, rows);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool inside = transposed ? k < K && r + e < rows : k + e < K;
            const float f = *reinterpret_cast<const float*>(base + (inside ? at + 4 * e : 0));   // the tile's first element otherwise
            v[e] = inside ? f : 0.f;
        }
        *reinterpret_cast<floatx4*>(dst + lane * 16) = floatx4{v[0], v[1], v[2], v[3]};
    };
    constexpr int J = JW_W + JW_X;
    auto request_piece = [&](int j, int t, char* stage) {
        if (j < JW_W) dma16(buf_w, off_w[j], t * step_w, stage + (NW * j + wave) * 1024);
        else dma16(buf_x, off_x[j - JW_W], t * step_x, stage + kX + (NW * (j - JW_W) + wave) * 1024);
    };
    auto request = [&](int t, int slot) {
        char* stage = ring + slot * kStage;
        if (t < full_tiles) {
#pragma unroll
            for (int j = 0; j < J; ++j) request_piece(j, t, stage);
        } else {
#pragma unroll
            for (int j = 0; j < JW_W; ++j) careful(WT, base_w, off_w[j], step_w, t, NW * j + wave, n0, N, stage + (NW * j + wave) * 1024);
#pragma unroll
            for (int j = 0; j < JW_X; ++j) careful(XT, base_x, off_x[j], step_x, t, NW * j + wave, m0, M, stage + kX + (NW * j + wave) * 1024);
        }
    };
    // Floats k = 8 g + 4 kh + {0..3} of row l32 of block `sub`.
    auto fragment = [&](auto transposed, const char* tile_base, int sub, int g) -> floatx4 {
        const char* block = tile_base + sub * 4096;
        if (!decltype(transposed)::value)
            return *reinterpret_cast<const floatx4*>(block + l32 * kRowBytes + (((2 * g + kh) ^ ((l32 >> 1) & 7)) << 4));
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int line = 4 * kh + e;   // of the eight of group g
            v[e] = *reinterpret_cast<const float*>(block + (8 * g + (line ^ ((line >> 2) & 1))) * 128 + l32 * 4);
        }
        return v;
    };

    floatx16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
    // Group i takes k-tiles t_begin + i, + KG, ...; all groups walk the same number of rounds, for the barriers.
    const int rounds = (t_end - t_begin + KG - 1) / KG;
    auto tile_at = [&](int r) { return t_begin + r * KG + group; };
#pragma unroll 1   // unrolled, the instructions of four requests are what a short product waits for
    for (int i = 0; i < STAGES; ++i)
        if (tile_at(i) < t_end) request(tile_at(i), i);
    // Requests up to tile r - 1 of this group have landed and this wavefront's LDS reads have returned; the `behind` tiles
    // from r on may be in flight if all went out as requests.
    auto landed = [&](int r, auto behind) {
        const int last = tile_at(r + decltype(behind)::value - 1);
        if (last < t_end && last < full_tiles)
            __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(decltype(behind)::value * J));
        else
            __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    floatx4 fw[4], fx[4];
    auto read_half = [&](int slot, auto half) {
        constexpr int g0 = decltype(half)::value * 2;
        const char* wt = ring + slot * kStage;
        const char* xt = wt + kX;
#pragma unroll
        for (int g = g0; g < g0 + 2; ++g) {
            fw[g] = fragment(std::integral_constant<bool, WT>{}, wt, sub_w, g);
            fx[g] = fragment(std::integral_constant<bool, XT>{}, xt, sub_x, g);
        }
        __builtin_amdgcn_sched_barrier(0);   // left alone, the compiler puts each pair in front of its MFMAs
    };
    auto multiply = [&](auto half, auto from, auto upto) {   // instructions [from, upto) of eight
        constexpr int g0 = decltype(half)::value * 2;
#pragma unroll
        for (int i = decltype(from)::value; i < decltype(upto)::value; ++i)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[g0 + i / 4][i % 4], fx[g0 + i / 4][i % 4], acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    typedef std::integral_constant<int, 0> First;
    typedef std::integral_constant<int, 1> Second;
    typedef std::integral_constant<int, 8> End;
    // Seven instructions on one half of a k-tile hide the reads of the other half, or of the first half of the next k-tile.
    // The one in front of the reads has waited for what came before them.
    landed(1, std::integral_constant<int, STAGES - 1>{});
    read_half(0, First{});
    int slot = 0, r = 0;
    // While all that is requested goes out as requests: nothing to decide, and an instruction's shadow has at most two of them.
    const int plain = (t_end < full_tiles ? t_end : full_tiles) - t_begin - group;   // tiles of the range, counted from the group's first
#pragma unroll 1
    for (; (r + STAGES) * KG < plain; ++r) {
        multiply(First{}, First{}, Second{});
        read_half(slot, Second{});
        multiply(First{}, Second{}, End{});
        __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((STAGES - 2) * J));   // tile r + 1 is readable, the slot of tile r free
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        char* const stage = ring + slot * kStage;
        slot = slot + 1 == STAGES ? 0 : slot + 1;
        multiply(Second{}, First{}, Second{});
        read_half(slot, First{});
#pragma unroll
        for (int i = 1; i < 8; ++i) {
#pragma unroll
            for (int j = (i - 1) * J / 7; j < i * J / 7; ++j) request_piece(j, tile_at(r + STAGES), stage);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[2 + i / 4][i % 4], fx[2 + i / 4][i % 4], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll 1
    for (; r < rounds; ++r) {
        if (KG > 1 && tile_at(r) >= t_end) break;   // the last round of a group that has one tile less
        multiply(First{}, First{}, Second{});
        read_half(slot, Second{});
        multiply(First{}, Second{}, End{});
        if (r + 1 < rounds) landed(r + 2, std::integral_constant<int, STAGES - 2>{});
        const int next = slot + 1 == STAGES ? 0 : slot + 1;
        multiply(Second{}, First{}, Second{});
        read_half(next, First{});   // behind the last tile what the slot holds, for nothing
        if (tile_at(r + STAGES) < t_end) request(tile_at(r + STAGES), slot);
        multiply(Second{}, Second{}, End{});
        slot = next;
    }
    // Lane holds row m = l32 and columns n = 8 g + 4 kh + {0..3} in acc[4 g + {0..3}].
    floatx4 quad[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) quad[g] = floatx4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    if (KG > 1) {   // the groups' sums meet in group 0, in the order of the groups
        __syncthreads();
        floatx4* fold = reinterpret_cast<floatx4*>(lds);
        if (group > 0) {
#pragma unroll
            for (int g = 0; g < 4; ++g) fold[(((group - 1) * NW + wave) * 4 + g) * 64 + lane] = quad[g];
        }
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int i = 0; i < KG - 1; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) quad[g] += fold[((i * NW + wave) * 4 + g) * 64 + lane];
    }
    if (splits > 1) {   // lane order, so that the partial sums are written and read in whole lines
        floatx4* dst = reinterpret_cast<floatx4*>(partial) + (static_cast<int64_t>(number) * NW + wave) * 256 + lane;
#pragma unroll
        for (int g = 0; g < 4; ++g) dst[g * 64] = quad[g];
        return;
    }
    const int64_t m = m0 + sub_x * 32 + l32;
    if (m >= M) return;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int64_t n = n0 + sub_w * 32 + 8 * g + 4 * kh;
        store_four(p.y + m * p.ldy + n, n, N, quad[g] + bias_of(p.bias, n, N));
    }
}

template <bool XT, bool WT, int NWM, int NWN, int KG, int STAGES>
__global__ __launch_bounds__(256) void gemm32_small(const Part32 p, int splits, float* __restrict__ partial) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    small_product<XT, WT, NWM, NWN, KG, STAGES>(p, blockIdx.x, splits, partial, lds);
}

// Sum of the splits' partial tiles and bias, workgroup `number`: a thread per quartet of columns.
template <int NWM, int NWN>
__device__ inline void sum_splits(const Part32& p, int splits, const float* __restrict__ partial, int number) {
    constexpr int NW = NWM * NWN;   // one workgroup per 32 x 32 block
    const int ntiles = p.tiles_m * p.tiles_n;
    const int tile = number / NW, wave = number - tile * NW;
    int tm, tn;
    tile_of_workgroup(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int64_t m = static_cast<int64_t>(tm) * (32 * NWM) + wave % NWM * 32 + (lane & 31);
    const int64_t n = static_cast<int64_t>(tn) * (32 * NWN) + wave / NWM * 32 + 8 * g + 4 * (lane >> 5);
    if (m >= p.M || n >= p.N) return;
    const floatx4* src = reinterpret_cast<const floatx4*>(partial) + static_cast<int64_t>(number) * 256 + threadIdx.x;
    const int64_t stride = static_cast<int64_t>(ntiles) * NW * 256;
    floatx4 s = {0.f, 0.f, 0.f, 0.f};
    int k = 0;
    for (; k + 4 <= splits; k += 4) {
        floatx4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = src[(k + u) * stride];
#pragma unroll
        for (int u = 0; u < 4; ++u) s += v[u];
    }
    for (; k < splits; ++k) s += src[k * stride];
    store_four(p.y + m * p.ldy + n, n, p.N, s + bias_of(p.bias, n, p.N));
}

template <int NWM, int NWN>
__global__ __launch_bounds__(256) void gemm32_small_sum(const Part32 p, int splits, const float* __restrict__ partial) {
    sum_splits<NWM, NWN>(p, splits, partial, blockIdx.x);
}

template <int NWM, int NWN>
int launch_sum(const Part32& part, int splits, const float* partial, hipStream_t s) {
    hipLaunchKernelGGL((gemm32_small_sum<NWM, NWN>), dim3(static_cast<uint32_t>(part.tiles_m * part.tiles_n * NWM * NWN)), dim3(256), 0, s, part, splits, partial);
    return check_launch("gemm32_small_sum");
}

template <bool XT, bool WT, int NWM, int NWN, int KG>
int launch(const char* who, Part32 part, int splits, float* partial, int dev, hipStream_t s) {
    static std::atomic<bool> reserved[kMaxDevices];   // the dynamic LDS size has been raised on that device (first use, any thread)
    constexpr int BM = 32 * NWM, BN = 32 * NWN, STAGES = 4, lds_bytes = KG * STAGES * (BM + BN) * kRowBytes;
    const auto kernel = gemm32_small<XT, WT, NWM, NWN, KG, STAGES>;
    if (lds_bytes > 65536 && !reserved[dev].load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        if (e != hipSuccess) return fail(static_cast<int>(e), "%s: cannot reserve %d bytes of LDS: %s", who, lds_bytes, hipGetErrorString(e));
        reserved[dev].store(true, std::memory_order_release);
    }
    part.tiles_m = static_cast<int>((part.M + BM - 1) / BM), part.tiles_n = static_cast<int>((part.N + BN - 1) / BN);
    const int ntiles = part.tiles_m * part.tiles_n;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(ntiles * splits)), dim3(256), lds_bytes, s, part, splits, partial);
    if (int rc = check_launch("gemm32_small")) return rc;
    return splits == 1 ? 0 : launch_sum<NWM, NWN>(part, splits, partial, s);
}

template <bool XT, bool WT>
int launch_shape(const char* who, const Small32& plan, const Part32& part, float* partial, int dev, hipStream_t s) {
    if (plan.groups == 4) return launch<XT, WT, 1, 1, 4>(who, part, plan.splits, partial, dev, s);
    if (plan.groups == 2) return launch<XT, WT, 1, 2, 2>(who, part, plan.splits, partial, dev, s);
    return launch<XT, WT, 2, 2, 1>(who, part, plan.splits, partial, dev, s);
}

// The adjoint of a linear shard in one launch: dx = dy . w and dw = dy^T . x in tiles of GX and GW groups, db = column sums of dy.
struct Adjoint32 {
    Part32 dx, dw;
    int splits_x, splits_w, blocks_x, blocks_w;   // workgroups of the products
    int first_w;                                  // dw's come first
    float *partial_x, *partial_w;
    float* db;
    int strips;
};

// By groups: wavefronts along m and n, stages (two workgroups per CU with one and two groups).
template <int G>
struct Shape32 {
    static constexpr int NWM = G == 1 ? 2 : 1, NWN = G == 4 ? 1 : 2, STAGES = G == 1 ? 4 : 3;
    static constexpr int kLds = G * STAGES * 32 * (NWM + NWN) * kRowBytes;
};

template <int GX, int GW>
__global__ __launch_bounds__(256) void linear32_adjoint(const Adjoint32 p) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    typedef Shape32<GX> X;
    typedef Shape32<GW> W;
    // Few strips of column sums come first, each a long chain of loads; many would keep the products waiting.
    const int products = p.blocks_x + p.blocks_w, first = p.strips <= kFirstStrips ? p.strips : 0;
    const int b = static_cast<int>(blockIdx.x) - first, x = p.first_w ? b - p.blocks_w : b, w = p.first_w ? b : b - p.blocks_x;
    if (b < 0 || b >= products)
        colsum_strip<2, 256, 4>(p.dx.x, p.dx.M, p.dx.K, p.dx.ldx, p.db, b < 0 ? blockIdx.x : b - products, p.strips, lds);
    else if (x >= 0 && x < p.blocks_x)
        small_product<false, true, X::NWM, X::NWN, GX, X::STAGES>(p.dx, x, p.splits_x, p.partial_x, lds);
    else
        small_product<true, true, W::NWM, W::NWN, GW, W::STAGES>(p.dw, w, p.splits_w, p.partial_w, lds);
}

template <int GX, int GW>
__global__ __launch_bounds__(256) void linear32_adjoint_sum(const Adjoint32 p, int blocks_x) {
    const int b = blockIdx.x;
    if (b < blocks_x) sum_splits<Shape32<GX>::NWM, Shape32<GX>::NWN>(p.dx, p.splits_x, p.partial_x, b);
    else sum_splits<Shape32<GW>::NWM, Shape32<GW>::NWN>(p.dw, p.splits_w, p.partial_w, b - blocks_x);
}

template <int GX, int GW>
int launch_adjoint(const Adjoint32& p, int dev, hipStream_t s) {
    static std::atomic<bool> reserved[kMaxDevices];
    typedef Shape32<GX> X;
    typedef Shape32<GW> W;
    constexpr int lds_bytes = X::kLds > W::kLds ? X::kLds : W::kLds;
    static_assert(colsum_lds_bytes(2, 256) <= lds_bytes, "the column sums do not fit");
    const auto kernel = linear32_adjoint<GX, GW>;
    if (lds_bytes > 65536 && !reserved[dev].load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        if (e != hipSuccess) return fail(static_cast<int>(e), "linear backward: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(e));
        reserved[dev].store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(p.blocks_x + p.blocks_w + p.strips)), dim3(256), lds_bytes, s, p);
    if (int rc = check_launch("linear32_adjoint")) return rc;
    const int sum_x = p.splits_x > 1 ? p.blocks_x / p.splits_x * X::NWM * X::NWN : 0, sum_w = p.splits_w > 1 ? p.blocks_w / p.splits_w * W::NWM * W::NWN : 0;
    if (sum_x + sum_w == 0) return 0;
    hipLaunchKernelGGL((linear32_adjoint_sum<GX, GW>), dim3(static_cast<uint32_t>(sum_x + sum_w)), dim3(256), 0, s, p, sum_x);
    return check_launch("linear32_adjoint_sum");
}

}  // namespace

// The estimates are fits to a sweep over M, N, K of 5 .. 16384 on all operand layouts, in microseconds: 4 + per k-tile (per
// round of one k-tile for every group) 0.68 for a lone 64 x 64 tile, 0.52 for each that a CU has to work through, 0.78 in
// two or four groups + the epilogue of every further tile + for splits a second launch (2.3, and 5 for
// what it and the workspace cost the host, which many callers wait for) and the partial tiles at 5 TB/s.
// They were fitted before the loop's halves overlapped, which takes 0.54, 0.48 and 0.57 where they say 0.68, 0.52 and 0.78; with
// those the choice is no better (4000 shapes, the product 1.02 times as fast and its adjoint as fast, single ones 0.6 to 1.6:
// fewer splits of long reductions, and products that linear_f32_split.hip has the lead in).
// Measured, general kernel of 128 x 128 tiles -> here: M 777, N 333, K 1024 107.2 -> 13.0 (two groups); M 8, N 4096, K 4096 365 -> 16.3.
Small32 plan_small32(int64_t M, int64_t N, int64_t K, int cus, int64_t workspace) {
    Small32 best;
    const int64_t ktiles = (K + BK - 1) / BK;
    double best_us = 1e30;
    for (const int groups : {1, 2, 4}) {
        const int64_t bm = groups == 1 ? 64 : 32, bn = groups == 4 ? 32 : 64, tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        if (tiles > 0xFFFFFF) continue;   // a launch has fewer than 2^32 threads, 256 per tile
        for (const int splits : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (splits > 1 && (tiles * splits > 4 * static_cast<int64_t>(cus) || ktiles < 2 * splits * groups || tiles * splits * bm * bn > workspace)) break;
            const int64_t per_cu = (tiles * splits + cus - 1) / cus, kt = (ktiles + splits - 1) / splits;
            double us = 4 + (splits > 1 ? 7.5 + static_cast<double>(tiles) * splits * bm * bn * 8 / 5e6 : 0);
            if (groups == 1)
                us += kt * (per_cu > 1 ? 0.52 * per_cu + 0.1 : 0.68) + (per_cu > 2 ? per_cu - 2 : 0) * 1.8;
            else
                us += ((kt + groups - 1) / groups) * 0.78 * per_cu + (per_cu - 1) * (groups == 2 ? 1.5 : 3.0);
            if (us >= best_us) continue;
            best_us = best.us = us;
            best.groups = groups, best.splits = splits, best.workspace = splits > 1 ? tiles * splits * bm * bn : 0;
        }
    }
    return best;
}

// Both products on one chip at the same time, next to `x` and `w`, how they are computed alone: a round of a workgroup (k-tiles of
// all its groups) is 0.52 us of its CU's matrix cores and at least 0.7 long.  No element is summed in fewer pieces than alone.
// The other way has 4.5 for the column sum, and 3 for each of the two further launches, of which 2 are the host's, where that may
// be what a step waits for.  All workgroups are resident at once: where there are more, the products fill the chip one by one.
AdjointPlan32 plan_adjoint32(int64_t M, int64_t N, int64_t K, bool want_db, int cus, int64_t workspace, const Small32& x, const Small32& w) {
    AdjointPlan32 best;
    if (!x.groups || x.edge || !w.groups || w.edge) return best;
    const double apart_us = x.us + w.us, launch_us = apart_us < 35 ? 3 : 1;
    double best_us = apart_us + (want_db ? 4.5 + launch_us : 0) + launch_us;
    double least_us = 3 + 4 * (static_cast<double>(M) * N + (static_cast<double>(M) + N) * K * 2) / 6e6;   // operands and results once
    if (want_db && 4 + M * 0.0032 > least_us) least_us = 4 + M * 0.0032;                                   // one strip of the column sums
    const double strips = want_db ? static_cast<double>((N + kNarrow - 1) / kNarrow) : 0;
    auto tiles = [](int64_t rows, int64_t cols, int g) {
        const int64_t bm = g == 1 ? 64 : 32, bn = g == 4 ? 32 : 64;
        return ((rows + bm - 1) / bm) * ((cols + bn - 1) / bn);
    };
    auto floats = [](int64_t blocks, int g) { return blocks * (g == 1 ? 4096 : g == 2 ? 2048 : 1024); };
    const int64_t kx = (N + BK - 1) / BK, kw = (M + BK - 1) / BK;
    for (const int gx : {1, 2, 4}) {
        for (const int gw : {1, 2, 4}) {
            const int64_t tiles_x = tiles(M, K, gx), tiles_w = tiles(N, K, gw), most = (gx == 4 || gw == 4 ? 1 : 2) * static_cast<int64_t>(cus);
            for (const int sx : {1, 2, 3, 4, 6, 8}) {
                if (tiles_x * sx > most || (sx > 1 && kx < 2 * sx * gx)) break;
                if (gx * sx < x.groups * x.splits) continue;
                for (const int sw : {1, 2, 3, 4, 6, 8}) {
                    const int64_t bx = tiles_x * sx, bw = tiles_w * sw, sums = (sx > 1 ? floats(bx, gx) : 0) + (sw > 1 ? floats(bw, gw) : 0);
                    if (bx + bw > most || (sw > 1 && kw < 2 * sw * gw)) break;
                    if (sums > workspace) break;
                    if (gw * sw < w.groups * w.splits) continue;
                    const int64_t nx = ((kx + sx - 1) / sx + gx - 1) / gx, nw = ((kw + sw - 1) / sw + gw - 1) / gw;
                    const double ex = gx == 1 ? 1.0 : gx == 2 ? 1.3 : 2.0, ew = gw == 1 ? 1.0 : gw == 2 ? 1.3 : 2.0;
                    const double all = (bx * (nx * 0.52 + ex) + bw * (nw * 0.52 + ew)) / cus * 1.1, longest = (nx > nw ? nx : nw) * 0.7;
                    double us = 4.5 + (all > longest ? all : longest) + strips / cus;
                    if (us < least_us) us = least_us;
                    if (sums) us += 5.5 + static_cast<double>(sums) * 8 / 5e6;
                    if (us >= best_us) continue;
                    best_us = us;
                    best.groups_x = gx, best.groups_w = gw, best.splits_x = sx, best.splits_w = sw, best.workspace = sums, best.first_w = nw > nx;
                }
            }
        }
    }
    return best;
}

int run_adjoint32(const AdjointPlan32& plan, const PartOf<float>& dx, const PartOf<float>& dw, float* db, float* workspace, hipStream_t s) {
    Adjoint32 p{};
    p.dx = dx, p.dw = dw, p.splits_x = plan.splits_x, p.splits_w = plan.splits_w, p.first_w = plan.first_w;
    auto tile = [](Part32& part, int g) {
        const int64_t bm = g == 1 ? 64 : 32, bn = g == 4 ? 32 : 64;
        part.tiles_m = static_cast<int>((part.M + bm - 1) / bm), part.tiles_n = static_cast<int>((part.N + bn - 1) / bn);
        return part.tiles_m * part.tiles_n;
    };
    p.blocks_x = tile(p.dx, plan.groups_x) * plan.splits_x, p.blocks_w = tile(p.dw, plan.groups_w) * plan.splits_w;
    p.partial_x = workspace;
    p.partial_w = workspace + (plan.splits_x > 1 ? static_cast<int64_t>(p.blocks_x) * (plan.groups_x == 1 ? 4096 : plan.groups_x == 2 ? 2048 : 1024) : 0);
    p.db = db, p.strips = db ? static_cast<int>((dx.K + kNarrow - 1) / kNarrow) : 0;
    int dev = 0;
    compute_units(dev);
    switch (plan.groups_x * 8 + plan.groups_w) {
        case 9: return launch_adjoint<1, 1>(p, dev, s);
        case 10: return launch_adjoint<1, 2>(p, dev, s);
        case 12: return launch_adjoint<1, 4>(p, dev, s);
        case 17: return launch_adjoint<2, 1>(p, dev, s);
        case 18: return launch_adjoint<2, 2>(p, dev, s);
        case 20: return launch_adjoint<2, 4>(p, dev, s);
        case 33: return launch_adjoint<4, 1>(p, dev, s);
        case 34: return launch_adjoint<4, 2>(p, dev, s);
        default: return launch_adjoint<4, 4>(p, dev, s);
    }
}

int run_small32(const char* who, const Small32& plan, bool xt, bool wt, const PartOf<float>& part, float* partial, int dev, hipStream_t s) {
    if (xt && wt) return launch_shape<true, true>(who, plan, part, partial, dev, s);
    if (xt) return launch_shape<true, false>(who, plan, part, partial, dev, s);
    if (wt) return launch_shape<false, true>(who, plan, part, partial, dev, s);
    return launch_shape<false, false>(who, plan, part, partial, dev, s);
}

int sum_small32(const PartOf<float>& part, int blocks, int splits, const float* partial, hipStream_t s) {
    return blocks == 2 ? launch_sum<2, 2>(part, splits, partial, s) : launch_sum<4, 4>(part, splits, partial, s);
}

}  // namespace ddl
