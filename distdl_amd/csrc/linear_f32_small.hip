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
#include "gemm_tiles.h"
#include "gemm32_small.h"
#include <type_traits>

namespace ddl {
namespace {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

constexpr int BK = kRowBytes / 4;   // floats of a k-tile
typedef PartOf<float> Part32;

template <bool XT, bool WT, int NWM, int NWN, int KG, int STAGES>
__global__ __launch_bounds__(256) void gemm32_small(const Part32 p, int splits, float* __restrict__ partial) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int NW = NWM * NWN, BM = 32 * NWM, BN = 32 * NWN;
    static_assert(NW * KG == 4, "four wavefronts per workgroup");
    constexpr int JW_W = BN / 8 / NW, JW_X = BM / 8 / NW;   // request instructions (1 KiB each) per wavefront and tile
    constexpr int kStage = (BM + BN) * kRowBytes, kX = BN * kRowBytes;   // a stage holds the w tile and then the x tile
    const int ntiles = p.tiles_m * p.tiles_n;
    const int split = static_cast<int>(blockIdx.x) / ntiles, tile = static_cast<int>(blockIdx.x) - split * ntiles;
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
    auto request = [&](int t, int slot) {
        char* stage = ring + slot * kStage;
        if (t < full_tiles) {
#pragma unroll
            for (int j = 0; j < JW_W; ++j) dma16(buf_w, off_w[j], t * step_w, stage + (NW * j + wave) * 1024);
#pragma unroll
            for (int j = 0; j < JW_X; ++j) dma16(buf_x, off_x[j], t * step_x, stage + kX + (NW * j + wave) * 1024);
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
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i)
        if (tile_at(i) < t_end) request(tile_at(i), i);
    int slot = 0;
#pragma unroll 1
    for (int r = 0; r < rounds; ++r) {
        // This wavefront's requests of tile r have landed (those of the STAGES - 2 tiles behind it may be in flight if all
        // went out as requests) and its LDS reads of tile r - 1 have returned: behind the barrier tile r is readable and
        // the slot of tile r - 1 is free.
        const int last = tile_at(r + STAGES - 2);
        if (last < t_end && last < full_tiles)
            __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((STAGES - 2) * (JW_W + JW_X)));
        else
            __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (tile_at(r + STAGES - 1) < t_end) request(tile_at(r + STAGES - 1), slot == 0 ? STAGES - 1 : slot - 1);
        if (KG > 1 && tile_at(r) >= t_end) continue;   // the last round of a group that has one tile less
        const char* wt = ring + slot * kStage;
        const char* xt = wt + kX;
        floatx4 fw[4], fx[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            fw[g] = fragment(std::integral_constant<bool, WT>{}, wt, sub_w, g);
            fx[g] = fragment(std::integral_constant<bool, XT>{}, xt, sub_x, g);
        }
        __builtin_amdgcn_sched_barrier(0);   // all reads first: left alone, the compiler puts each pair in front of its MFMAs
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[g][e], fx[g][e], acc, 0, 0, 0);
        slot = slot + 1 == STAGES ? 0 : slot + 1;
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
        floatx4* dst = reinterpret_cast<floatx4*>(partial) + (static_cast<int64_t>(blockIdx.x) * NW + wave) * 256 + lane;
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

// Sum of the splits' partial tiles and bias.  A thread per quartet of columns.
template <int NWM, int NWN>
__global__ __launch_bounds__(256) void gemm32_small_sum(const Part32 p, int splits, const float* __restrict__ partial) {
    constexpr int NW = NWM * NWN;   // one workgroup per 32 x 32 block
    const int ntiles = p.tiles_m * p.tiles_n;
    const int tile = static_cast<int>(blockIdx.x) / NW, wave = static_cast<int>(blockIdx.x) - tile * NW;
    int tm, tn;
    tile_of_workgroup(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int64_t m = static_cast<int64_t>(tm) * (32 * NWM) + wave % NWM * 32 + (lane & 31);
    const int64_t n = static_cast<int64_t>(tn) * (32 * NWN) + wave / NWM * 32 + 8 * g + 4 * (lane >> 5);
    if (m >= p.M || n >= p.N) return;
    const floatx4* src = reinterpret_cast<const floatx4*>(partial) + static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
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

}  // namespace

// The estimates are fits to a sweep over M, N, K of 5 .. 16384 on all operand layouts, in microseconds: 4 + per k-tile (per
// round of one k-tile for every group) 0.68 for a lone 64 x 64 tile, 0.52 for each that a CU has to work through, 0.78 in
// two or four groups + the epilogue of every further tile + for splits a second launch (2.3, and 5 for
// what it and the workspace cost the host, which many callers wait for) and the partial tiles at 5 TB/s.
// Measured, general kernel of 128 x 128 tiles -> here: M 777, N 333, K 1024 107.2 -> 17.7 (two groups; 15.7 in three
// splits, which the host's share makes the slower call); its adjoint M 777, N 1024, K 333 45.4 -> 12.4 and M 333, N 1024, K 777, both operands along their rows, 84.1 ->
// 15.6; M 8, N 4096, K 4096 365 -> 20.
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
