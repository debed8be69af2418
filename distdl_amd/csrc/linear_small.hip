// DistributedLinear shard products in 16 bits that large tiles leave most of the
// chip idle for: y[M,N] = a[M,K] . b[N,K]^T + bias[N], as in linear_gemm.hip
// (same operand layouts, fp32 accumulation, one rounding to the result's type).
//
// gemm16_skinny (M up to 64, both operands contiguous along k: a decode step).
//   Bound by streaming w from HBM: M 8, N 3584, K 8192 takes 13.1 us (69.0 in large
//   tiles), of which 10 are w's 58.7 MB at 5.9 TB/s.  A workgroup owns 16 columns and
//   all rows; its eight wavefronts split the reduction, each with a ring of its own in
//   LDS, so that the loop has no barrier and some 100 KiB of requests are in flight
//   per CU; the eight partial sums meet in LDS in the order of the wavefronts.
//   Requests into LDS, because loads into registers reach a third of their rate on
//   one CU (N 64, K 8192: 6.7 us, through registers 13.4); 32 columns per workgroup
//   halve the reads of x but leave CUs idle (21 us at N 3584).
//
// gemm16_small (tiles of 64 x 64, k-tiles of 64).
//   Bound by LDS (a k-tile is 32 KiB of fragment reads and 16 KiB of requests, 384
//   cycles next to 128 of MFMA; 0.19 us = 456 measured) and by how many CUs have work.
//   Tiles are staged like in linear_gemm.hip (global -> LDS requests, the same
//   swizzles, transposing LDS reads) through a ring of four stages; two workgroups,
//   or two groups of wavefronts of one workgroup that take alternate k-tiles, share a
//   CU and hide each other's waits, so the loop itself is plain: wait for tile t,
//   barrier, request tile t + 3, multiply.  Tiles of 128 x 128 (one workgroup per CU)
//   took 0.51 us per k-tile whatever the shape, no better than large tiles.  Where
//   even these tiles are too few, the reduction is split over `splits` workgroups per
//   tile; their fp32 sums go through a workspace and gemm16_small_sum adds them in the
//   order of the splits.
#include "gemm16_parts.h"
#include <type_traits>

namespace ddl {
namespace {

constexpr int BK = kRowBytes / 2;   // 16-bit elements of a k-tile

// ---- up to 64 rows ---------------------------------------------------------

constexpr int kSkinnyWaves = 8;

// XP: 8-row pieces of x (M <= 8 XP).  A step is 64 k: 128 bytes of 16 rows of w and of the rows of x.
template <int XP>
struct Skinny {
    static constexpr int kStep = (2 + XP) * 1024;                              // bytes of a step in LDS: w, then x
    static constexpr int kStages = XP == 1 ? 6 : XP == 2 ? 4 : XP == 4 ? 3 : 2;   // steps of a wavefront's ring
    static constexpr int kLds = kSkinnyWaves * kStages * kStep;
    static constexpr int TM = XP == 1 ? 1 : XP / 2;
};

template <bool F16, int XP>
__global__ __launch_bounds__(kSkinnyWaves * 64) void gemm16_skinny(const Part16 p) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    typedef Skinny<XP> S;
    constexpr int TM = S::TM, J = 2 + XP;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, kg = lane >> 4;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * 16;
    const int64_t M = p.M, N = p.N, K = p.K;

    // Request j of a step: rows 8 j .. + 7 of w (j < 2) or 8 (j - 2) .. of x, one 128-byte line per eight lanes, chunks
    // swizzled by row as in linear_gemm.hip.  Rows past the end repeat the last one; their products are not stored.
    const char* const base_w = reinterpret_cast<const char*>(p.w + n0 * p.ldw);
    const char* const base_x = reinterpret_cast<const char*>(p.x);
    const u32x4 buf_w = raw_buffer(base_w), buf_x = raw_buffer(base_x);
    int off[J], chunk[J];   // byte offset of this lane's chunk; its first k inside a step
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int row = (j < 2 ? j : j - 2) * 8 + (lane >> 3);
        const int64_t rows = j < 2 ? N - n0 : M;
        chunk[j] = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
        off[j] = static_cast<int>(((row < rows ? row : rows - 1) * (j < 2 ? p.ldw : p.ldx) + chunk[j]) * 2);
    }
    const int steps = static_cast<int>((K + BK - 1) / BK), full = static_cast<int>(K / BK);
    char* const ring = lds + wave * (S::kStages * S::kStep);
    auto request = [&](int s, int slot) {
        char* stage = ring + slot * S::kStep;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (s < full) {
                dma16(j < 2 ? buf_w : buf_x, off[j], s * (BK * 2), stage + j * 1024);
            } else {   // the step that straddles K goes through registers, zeros past K
                uint4 v = make_uint4(0, 0, 0, 0);
                if (static_cast<int64_t>(s) * BK + chunk[j] < K)
                    v = *reinterpret_cast<const uint4*>((j < 2 ? base_w : base_x) + off[j] + static_cast<int64_t>(s) * (BK * 2));
                *reinterpret_cast<uint4*>(stage + j * 1024 + lane * 16) = v;
            }
        }
    };

    floatx4 acc[TM];
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    // Wavefront v takes steps v, v + 8, ...; its ring is its own, so no barrier is needed.
    constexpr int kAhead = S::kStages - 1;
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
        if (wave + i * kSkinnyWaves < steps) request(wave + i * kSkinnyWaves, i);
    const int row_x = XP == 1 ? l16 & 7 : l16;
    int slot = 0;
#pragma unroll 1
    for (int s = wave; s < steps; s += kSkinnyWaves) {
        // Step s has landed (the kAhead - 1 steps behind it may be in flight if all went out as requests) and this
        // wavefront's reads of the step before have returned.
        if (s + (kAhead - 1) * kSkinnyWaves < full)
            __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((kAhead - 1) * J));
        else
            __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
        asm volatile("" ::: "memory");
        if (s + kAhead * kSkinnyWaves < steps) request(s + kAhead * kSkinnyWaves, slot == 0 ? S::kStages - 1 : slot - 1);
        const char* wt = ring + slot * S::kStep;
        const char* xt = wt + 2048;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const bf16x8 fw = *reinterpret_cast<const bf16x8*>(wt + l16 * kRowBytes + (((4 * ks + kg) ^ ((l16 >> 1) & 7)) << 4));
#pragma unroll
            for (int b = 0; b < TM; ++b) {
                const bf16x8 fx = *reinterpret_cast<const bf16x8*>(xt + (b * 16 + row_x) * kRowBytes + (((4 * ks + kg) ^ ((row_x >> 1) & 7)) << 4));
                acc[b] = mfma<F16>(fw, fx, acc[b]);
            }
        }
        slot = slot + 1 == S::kStages ? 0 : slot + 1;
    }
    __syncthreads();   // the rings are free
    floatx4* sums = reinterpret_cast<floatx4*>(lds);   // [wave][16-row block][lane]
#pragma unroll
    for (int b = 0; b < TM; ++b) sums[(wave * TM + b) * 64 + lane] = acc[b];
    __syncthreads();
    // One element per thread and round: 16-row block b, lane l, column 4 (l / 16) + e of row l % 16.
    for (int i = threadIdx.x; i < TM * 256; i += kSkinnyWaves * 64) {
        const int b = i >> 8, l = (i >> 2) & 63, e = i & 3;
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < kSkinnyWaves; ++k) v += sums[(k * TM + b) * 64 + l][e];
        const int64_t m = b * 16 + (l & 15), n = n0 + 4 * (l >> 4) + e;
        if (m < M && n < N) {
            if (p.bias) v += elem_to_f32<F16>(p.bias[n]);
            p.y[m * p.ldy + n] = f32_to_elem<F16>(v);
        }
    }
}

// ---- small tiles -----------------------------------------------------------

template <bool F16, bool XT, bool WT, int NWM, int NWN, int TM, int TN, int STAGES, int KG>
__global__ __launch_bounds__(KG * NWM * NWN * 64) void gemm16_small(const Part16 p, int splits, float* __restrict__ partial) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int NW = NWM * NWN, BM = 16 * NWM * TM, BN = 16 * NWN * TN;
    constexpr int JW_W = BN / 8 / NW, JW_X = BM / 8 / NW;   // request instructions (1 KiB each) per wavefront and tile
    static_assert(JW_W * 8 * NW == BN && JW_X * 8 * NW == BM && BM % 64 == 0 && BN % 64 == 0, "tile does not divide among the wavefronts");
    constexpr int kStage = (BM + BN) * kRowBytes, kX = BN * kRowBytes;   // a stage holds the w tile and then the x tile
    const int ntiles = p.tiles_m * p.tiles_n;
    const int split = static_cast<int>(blockIdx.x) / ntiles, tile = static_cast<int>(blockIdx.x) - split * ntiles;
    int tm, tn;
    tile_of_workgroup(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int64_t M = p.M, N = p.N, K = p.K;
    const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
    const int lane = threadIdx.x & 63, group = __builtin_amdgcn_readfirstlane(threadIdx.x / (NW * 64));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) - group * NW;   // inside its group
    const int l16 = lane & 15, kg = lane >> 4;
    const int sub_w = (wave / NWM) * TN, sub_x = (wave % NWM) * TM;   // first 16-row block of this wavefront in the w and x tiles

    // k-tiles [t, t_end) of this workgroup
    const int ktiles = static_cast<int>((K + BK - 1) / BK), full_tiles = static_cast<int>(K / BK);
    const int per = (ktiles + splits - 1) / splits;
    const int t_begin = split * per < ktiles ? split * per : ktiles, t_end = t_begin + per < ktiles ? t_begin + per : ktiles;

    char* const ring = lds + group * (STAGES * kStage);

    // Requests: 1 KiB piece i = NW j + wave of a tile.  Contiguous along k: rows 8 i .. + 7.  Contiguous along the rows:
    // k-lines 8 (i % 8) .. + 7 of panel i / 8 (64 rows).  Swizzles, clamps and byte offsets as in linear_gemm.hip.
    const char* const base_w = reinterpret_cast<const char*>(WT ? p.w + n0 : p.w + n0 * p.ldw);
    const char* const base_x = reinterpret_cast<const char*>(XT ? p.x + m0 : p.x + m0 * p.ldx);
    const u32x4 buf_w = raw_buffer(base_w), buf_x = raw_buffer(base_x);
    const int step_w = WT ? static_cast<int>(p.ldw) * (BK * 2) : BK * 2;
    const int step_x = XT ? static_cast<int>(p.ldx) * (BK * 2) : BK * 2;
    // first k (contiguous along k) or k-line of this lane's chunk of piece i inside a k-tile
    auto chunk_k = [&](bool transposed, int i) {
        const int row = i * 8 + (lane >> 3);
        return transposed ? 8 * (i & 7) + (lane >> 3) : ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    };
    auto lane_offset = [&](bool transposed, int i, int64_t origin, int64_t rows, int64_t ld) -> int {
        const int k = chunk_k(transposed, i);
        if (!transposed) {
            const int row = i * 8 + (lane >> 3);
            const int64_t rr = origin + row < rows ? row : rows - 1 - origin;
            return static_cast<int>((rr * ld + k) * 2);
        }
        const int h = ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
        int col = (i >> 3) * 64 + ((lane & 7) ^ (h << 1)) * 8;
        if (origin + col >= rows) col = 0;
        return static_cast<int>((k * ld + col) * 2);
    };
    int off_w[JW_W], off_x[JW_X];
#pragma unroll
    for (int j = 0; j < JW_W; ++j) off_w[j] = lane_offset(WT, NW * j + wave, n0, N, p.ldw);
#pragma unroll
    for (int j = 0; j < JW_X; ++j) off_x[j] = lane_offset(XT, NW * j + wave, m0, M, p.ldx);
    auto request = [&](int t, int slot) {
        char* stage = ring + slot * kStage;
        if (t < full_tiles) {
#pragma unroll
            for (int j = 0; j < JW_W; ++j) dma16(buf_w, off_w[j], t * step_w, stage + (NW * j + wave) * 1024);
#pragma unroll
            for (int j = 0; j < JW_X; ++j) dma16(buf_x, off_x[j], t * step_x, stage + kX + (NW * j + wave) * 1024);
        } else {   // the tile that straddles K goes through registers, zeros past K
#pragma unroll
            for (int j = 0; j < JW_W; ++j) {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (static_cast<int64_t>(t) * BK + chunk_k(WT, NW * j + wave) < K)
                    v = *reinterpret_cast<const uint4*>(base_w + off_w[j] + static_cast<int64_t>(t) * step_w);
                *reinterpret_cast<uint4*>(stage + (NW * j + wave) * 1024 + lane * 16) = v;
            }
#pragma unroll
            for (int j = 0; j < JW_X; ++j) {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (static_cast<int64_t>(t) * BK + chunk_k(XT, NW * j + wave) < K)
                    v = *reinterpret_cast<const uint4*>(base_x + off_x[j] + static_cast<int64_t>(t) * step_x);
                *reinterpret_cast<uint4*>(stage + kX + (NW * j + wave) * 1024 + lane * 16) = v;
            }
        }
    };

    // Fragment reads: as in linear_gemm.hip.
    const int tr_lane = (8 * kg + (l16 >> 2)) * 128 + (l16 & 3) * 8;
    const int tr_h = (((l16 >> 3) & 1) | ((kg & 1) << 1)) << 5;
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef short short8v __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) short4v* lds_short4;
    auto fragment = [&](auto transposed, const char* tile_base, int sub, int ks) -> bf16x8 {
        bf16x8 out;
        if (decltype(transposed)::value) {
            const char* q = tile_base + (sub >> 2) * 8192 + ks * (32 * 128) + (tr_lane + (((sub & 3) << 5) ^ tr_h));
            const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(q));
            const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(q + 4 * 128));
            const short8v both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            __builtin_memcpy(&out, &both, 16);
        } else {
            out = *reinterpret_cast<const bf16x8*>(tile_base + sub * (16 * kRowBytes) + l16 * kRowBytes + (((4 * ks + kg) ^ ((l16 >> 1) & 7)) << 4));
        }
        return out;
    };

    floatx4 acc[TN][TM];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};

    // Group g takes k-tiles t_begin + g, + KG, ...; all groups walk the same number of rounds, for the barriers.
    const int rounds = (t_end - t_begin + KG - 1) / KG;
    auto tile_at = [&](int r) { return t_begin + r * KG + group; };
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i)
        if (tile_at(i) < t_end) request(tile_at(i), i);
    int slot = 0;
#pragma unroll 1
    for (int r = 0; r < rounds; ++r) {
        // This wavefront's requests of tile r have landed: those of the STAGES - 2 tiles behind it may be in flight if all of
        // them went out as requests (otherwise wait for everything).  Its LDS reads of tile r - 1 have returned as well, so
        // behind the barrier tile r is readable and the slot of tile r - 1 is free.
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
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8 fw[TN], fx[TM];
#pragma unroll
            for (int a = 0; a < TN; ++a) fw[a] = fragment(std::integral_constant<bool, WT>{}, wt, sub_w + a, ks);
#pragma unroll
            for (int b = 0; b < TM; ++b) fx[b] = fragment(std::integral_constant<bool, XT>{}, xt, sub_x + b, ks);
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b) acc[a][b] = mfma<F16>(fw[a], fx[b], acc[a][b]);
        }
        slot = slot + 1 == STAGES ? 0 : slot + 1;
    }
    if (KG > 1) {   // the groups' sums meet in group 0, in the order of the groups
        __syncthreads();
        floatx4* fold = reinterpret_cast<floatx4*>(lds);
        if (group > 0) {
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b) fold[(((group - 1) * NW + wave) * (TN * TM) + a * TM + b) * 64 + lane] = acc[a][b];
        }
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int g = 0; g < KG - 1; ++g)
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b) acc[a][b] += fold[((g * NW + wave) * (TN * TM) + a * TM + b) * 64 + lane];
    }

    if (splits > 1) {   // lane order, so that the partial sums are written and read in whole lines
        floatx4* dst = reinterpret_cast<floatx4*>(partial) + (static_cast<int64_t>(blockIdx.x) * NW + wave) * (TN * TM * 64) + lane;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) dst[(a * TM + b) * 64] = acc[a][b];
        return;
    }
#pragma unroll
    for (int a = 0; a < TN; ++a) {
        const int64_t n = n0 + (sub_w + a) * 16 + 4 * kg;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < N) bv[e] = elem_to_f32<F16>(p.bias[n + e]);
        }
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            const int64_t m = m0 + (sub_x + b) * 16 + l16;
            if (m >= M) continue;
            const float v[4] = {acc[a][b][0] + bv[0], acc[a][b][1] + bv[1], acc[a][b][2] + bv[2], acc[a][b][3] + bv[3]};
            store_four<F16>(p.y, p.ldy, m, n, N, v);
        }
    }
}

constexpr int kStages = 4;

// Kernel functions whose dynamic LDS size has been raised on a device (first use, any thread): a flag per instantiation.
template <typename Kernel>
int reserve_lds(const char* who, Kernel kernel, std::atomic<bool> (&reserved)[kMaxDevices], int dev, int bytes) {
    if (bytes <= 65536 || reserved[dev].load(std::memory_order_acquire)) return 0;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(static_cast<int>(e), "%s: cannot reserve %d bytes of LDS: %s", who, bytes, hipGetErrorString(e));
    reserved[dev].store(true, std::memory_order_release);
    return 0;
}

template <bool F16, int XP>
int launch_skinny(const char* who, const Part16& part, int dev, hipStream_t s) {
    static std::atomic<bool> reserved[kMaxDevices];
    if (int rc = reserve_lds(who, gemm16_skinny<F16, XP>, reserved, dev, Skinny<XP>::kLds)) return rc;
    hipLaunchKernelGGL((gemm16_skinny<F16, XP>), dim3(static_cast<uint32_t>((part.N + 15) / 16)), dim3(kSkinnyWaves * 64), Skinny<XP>::kLds, s, part);
    return check_launch("gemm16_skinny");
}

template <bool F16, bool XT, bool WT, int NWM, int NWN, int TM, int TN, int KG>
int launch_small(const char* who, const Part16& part, int splits, float* partial, int dev, hipStream_t s) {
    static std::atomic<bool> reserved[kMaxDevices];
    constexpr int BM = 16 * NWM * TM, BN = 16 * NWN * TN, lds_bytes = KG * kStages * (BM + BN) * kRowBytes;
    const auto kernel = gemm16_small<F16, XT, WT, NWM, NWN, TM, TN, kStages, KG>;
    if (int rc = reserve_lds(who, kernel, reserved, dev, lds_bytes)) return rc;
    const int ntiles = part.tiles_m * part.tiles_n;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(ntiles * splits)), dim3(KG * NWM * NWN * 64), lds_bytes, s, part, splits, partial);
    if (int rc = check_launch("gemm16_small")) return rc;
    if (splits == 1) return 0;
    hipLaunchKernelGGL((gemm16_small_sum<F16, NWM, NWN, TM, TN>), dim3(static_cast<uint32_t>(ntiles * (BM * BN / 1024))), dim3(256), 0, s, part,
                       splits, static_cast<const float*>(partial));
    return check_launch("gemm16_small_sum");
}

template <bool F16, bool XT, bool WT>
int launch_kind(const char* who, const Small16& plan, Part16 part, float* partial, int dev, hipStream_t s) {
    part.tiles_m = static_cast<int>((part.M + 63) / 64), part.tiles_n = static_cast<int>((part.N + 63) / 64);
    if (plan.groups == 2) return launch_small<F16, XT, WT, 2, 2, 2, 2, 2>(who, part, plan.splits, partial, dev, s);
    return launch_small<F16, XT, WT, 2, 2, 2, 2, 1>(who, part, plan.splits, partial, dev, s);
}

template <bool F16>
int launch16(const char* who, const Small16& plan, bool xt, bool wt, const Part16& part, float* partial, int dev, hipStream_t s) {
    if (plan.kind == Small16::kSkinny) {
        if (part.M > 32) return launch_skinny<F16, 8>(who, part, dev, s);
        if (part.M > 16) return launch_skinny<F16, 4>(who, part, dev, s);
        if (part.M > 8) return launch_skinny<F16, 2>(who, part, dev, s);
        return launch_skinny<F16, 1>(who, part, dev, s);
    }
    if (xt && wt) return launch_kind<F16, true, true>(who, plan, part, partial, dev, s);
    if (xt) return launch_kind<F16, true, false>(who, plan, part, partial, dev, s);
    if (wt) return launch_kind<F16, false, true>(who, plan, part, partial, dev, s);
    return launch_kind<F16, false, false>(who, plan, part, partial, dev, s);
}

}  // namespace

// The estimates are fits to a sweep over M, N, K of 8 .. 28672 on all four operand layouts (within 10 % where it
// matters), in microseconds:
//   skinny   3 + what takes longest: a workgroup's bytes at the 110 GB/s that requests into one CU's LDS reach, all
//            workgroups' bytes at 15 TB/s (the L2s), w once at 6 TB/s (HBM)
//   tiles    3.8 + per k-tile 0.19 for each tile a CU has (0.30 for a lone workgroup, whose waits nothing hides;
//            0.375 per pair of k-tiles with two groups, which hide each other's) + 1.4 for the epilogue of every tile
//            beyond those resident at the start
//   splits   2.3 for the second launch and 5 for what it and the workspace cost the host, which many callers wait for
//            (M 6964, N 136, K 5632: 39.5 in two splits, 38 without) + the partial tiles (16 KiB, written and read) at 5 TB/s
// Measured, large tiles -> here: M 8, N 3584, K 8192 69.0 -> 13.1 us (skinny; 14.2 as tiles in two groups and four splits);
// M 64 of the same 69.5 -> 15.4 (two groups, four splits; 20.7 skinny); M 1024, N 1024, K 4096 (x w^T with w read down its
// columns) 39.1 -> 19.5 (two groups; 21.4 in two splits); M 1024, N 512, K 512 10.8 -> 6.0.  Large tiles stay where they
// fill the chip: M 1024, N 4096, K 1024 16.3, here 20.3.
Small16 plan_small16(bool xt, bool wt, int64_t M, int64_t N, int64_t K, int cus, int64_t workspace, double large_us) {
    Small16 best;
    const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64), ktiles = (K + BK - 1) / BK;
    const double hbm_us = (static_cast<double>(M) + N) * K * 2 / 6e6 + 3;   // both operands once
    double best_us = large_us * 0.92;   // what the fits are unsure of
    auto take = [&](double us, Small16::Kind kind, int groups, int splits) {
        if (us < hbm_us) us = hbm_us;
        if (us >= best_us) return;
        best_us = best.us = us;
        best.kind = kind, best.groups = groups, best.splits = splits, best.workspace = splits > 1 ? tiles * splits * 4096 : 0;
    };
    if (M <= 64 && !xt && !wt && N <= 0x7FFFFF) {
        const int64_t workgroups = (N + 15) / 16, pieces = M > 32 ? 8 : M > 16 ? 4 : M > 8 ? 2 : 1;
        const double bytes = static_cast<double>(ktiles) * (2 + pieces) * 1024;
        const double cu = static_cast<double>((workgroups + cus - 1) / cus) * bytes / 110e3, l2 = workgroups * bytes / 15e6;
        take(3 + (cu > l2 ? cu : l2), Small16::kSkinny, 1, 1);
    }
    if (tiles > 16 * static_cast<int64_t>(cus)) return best;
    for (const int splits : {1, 2, 3, 4, 6, 8, 12, 16}) {
        if (splits > 1 && (tiles * splits > 4 * static_cast<int64_t>(cus) || ktiles < 4 * splits || tiles * splits * 4096 > workspace)) break;
        const int64_t per_cu = (tiles * splits + cus - 1) / cus, kt = (ktiles + splits - 1) / splits;
        const double sum = splits > 1 ? 7.5 + tiles * splits * 0.0066 : 0;
        const double step = per_cu > 1 ? 0.19 * per_cu : 0.30;
        take(3.8 + kt * step + (per_cu > 2 ? per_cu - 2 : 0) * 1.4 + sum, Small16::kTiles, 1, splits);
        take(3.9 + ((kt + 1) / 2) * 0.375 * per_cu + (per_cu - 1) * 1.4 + sum, Small16::kTiles, 2, splits);
    }
    return best;
}

int run_small16(const char* who, const Small16& plan, bool f16, bool xt, bool wt, const Part16& part, float* partial, int dev, hipStream_t s) {
    return f16 ? launch16<true>(who, plan, xt, wt, part, partial, dev, s) : launch16<false>(who, plan, xt, wt, part, partial, dev, s);
}

}  // namespace ddl
