// 16-bit products of operands at any address and pitch, for sizes that the large
// tiles and the copies they need in front of them are too much for:
// y[M,N] = a[M,K] . b[N,K]^T + bias[N], operand layouts and arithmetic as in
// linear_gemm.hip (fp32 accumulation, one rounding to the result's type).
//
// gemm16_any (tiles of 64 x 64 or 128 x 128, k-tiles of 64, four wavefronts).
//   Requests into LDS want 4-byte alignment, so a tile comes through registers, 16
//   bytes a lane at any address, and goes into LDS in the layouts of linear_gemm.hip.
//   Bound by a k-tile's latencies while a CU has one workgroup and by LDS and the L1
//   when it has more: what matters is that loads stay in flight.  So the loop has no
//   branch and no masked load: tile i + 2 is requested while tile i is multiplied, one
//   barrier per k-tile, the LDS writes of tile i + 1 between the MFMAs of the second
//   half.  A tile that needs care (K ends in it, or its last chunk would run past the
//   operand) is taken first: its pieces are read from where they still lie inside and
//   shifted (drop), once, ahead of the loop.  With that care inside the loop the
//   compiler waits for every load in flight.  M 2276, N 456, K 3299 (training step of
//   the all-gather linear layer): y 46.3 -> 24.8 us, dx 36.6 -> 20.5, dw 28.4 -> 24.1;
//   M 564, N 1060, K 6838: 30.8 -> 25.9, 29.5 -> 23.5, 39.1 -> 18.2.
//   Tiles of 128 x 128 move half the bytes per flop (0.6 us per k-tile and CU against
//   1.0 for four of 64 x 64), smaller ones fill the chip: see plan_any16.
//
// linear16_adjoint (dx, dw and db of a linear shard).
//   Bound by launches and by CUs that have nothing to do: each of the three leaves most of the
//   chip idle when it is small, and waits for the one before.  Workgroups of all of them in one
//   launch, the product with the longer workgroups first: M 336, N 77, K 603 bf16 14.6 -> 5.7 us,
//   M 120, N 2258, K 3584 41.7 -> 15.4, M 718, N 821, K 5156 60.2 -> 32.8, M 1024, N 4096, K 1024
//   (aligned, before: requests into LDS, tiles of 128 x 256) 38.3 -> 30.0.  See plan_adjoint16.
//
// gemm16_thin (K below 8, at least one operand read along k).
//   A reduction shorter than a 16-byte load.  Bound by the result's stores; an output
//   element per lane.
#include "colsum.h"
#include "gemm16_parts.h"
#include <type_traits>

namespace ddl {
namespace {

constexpr int BK = kRowBytes / 2;   // 16-bit elements of a k-tile
constexpr int kAnyThreads = 256;

// The eight elements of `v` from number `s` on, zeros behind them.
__device__ inline uint4 drop(uint4 v, int s) {
    uint32_t w[5] = {v.x, v.y, v.z, v.w, 0};
    if (s & 4) w[0] = w[2], w[1] = w[3], w[2] = 0, w[3] = 0;
    if (s & 2) w[0] = w[1], w[1] = w[2], w[2] = w[3], w[3] = 0;
    if (s & 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = (w[e] >> 16) | (w[e + 1] << 16);
    }
    if (s >= 8) w[0] = w[1] = w[2] = w[3] = 0;
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// Workgroup `block` of the tiles_m x tiles_n x splits of a product: tiles of 64 T x 64 T, a wavefront has 32 T x 32 T.
template <bool F16, bool XT, bool WT, int T>
__device__ __forceinline__ void any_product(const Part16& p, int block, int splits, float* __restrict__ partial, char* lds) {
    constexpr int NWM = 2, TM = 2 * T, TN = 2 * T, NW = 4, J = 2 * T, B = 64 * T;   // J: 1 KiB pieces per wavefront and operand
    constexpr int kStage = 2 * B * kRowBytes, kX = B * kRowBytes;
    const int ntiles = p.tiles_m * p.tiles_n;
    const int split = block / ntiles, tile = block - split * ntiles;
    int tm, tn;
    tile_of_workgroup(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int64_t M = p.M, N = p.N, K = p.K, m0 = static_cast<int64_t>(tm) * B, n0 = static_cast<int64_t>(tn) * B;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, kg = lane >> 4;
    const int sub_w = (wave / NWM) * TN, sub_x = (wave % NWM) * TM;

    // k-tiles [t_begin, t_end) of this split.  The last one of all needs care where K ends in it, or where an operand read
    // along its rows has a chunk there that would run over into a k-line which the last one has not.
    const int ktiles = static_cast<int>((K + BK - 1) / BK);
    const int full_tiles = static_cast<int>(((WT && N % 8 != 0) || (XT && M % 8 != 0) ? K - 1 : K) / BK);
    const int per = (ktiles + splits - 1) / splits;
    const int t_begin = split * per < ktiles ? split * per : ktiles, t_end = t_begin + per < ktiles ? t_begin + per : ktiles;
    const int n = t_end - t_begin, has_tail = n > 0 && t_end > full_tiles ? 1 : 0;

    const uint16_t* const base_w = WT ? p.w + n0 : p.w + n0 * p.ldw;
    const uint16_t* const base_x = XT ? p.x + m0 : p.x + m0 * p.ldx;
    const int64_t step_w = WT ? p.ldw * BK : BK, step_x = XT ? p.ldx * BK : BK;   // elements from one k-tile to the next
    // Where this lane's chunk of piece i lies, from the tile's first row and k-tile 0 on: swizzles as in linear_gemm.hip, rows
    // past the end repeat the last one, chunks past it the first of the tile.
    auto row_of = [&](int i) { return i * 8 + (lane >> 3); };
    auto first_k = [&](int i) { return ((lane & 7) ^ ((row_of(i) >> 1) & 7)) * 8; };
    auto line_of = [&](int i) { return 8 * (i & 7) + (lane >> 3); };
    auto first_row = [&](int i, int64_t left) -> int64_t {
        const int k = line_of(i), h = ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
        const int col = (i >> 3) * 64 + ((lane & 7) ^ (h << 1)) * 8;
        return col < left ? col : 0;
    };
    auto place = [&](bool transposed, int i, int64_t left, int64_t ld) -> int64_t {   // left: rows of the operand from the tile's first on
        if (transposed) return line_of(i) * ld + first_row(i, left);
        return (row_of(i) < left ? row_of(i) : left - 1) * ld + first_k(i);
    };
    // The same in the tile that needs care: moved back to where 16 bytes still lie inside the operand, by `s` elements; 8 for
    // a chunk that is all zeros.
    auto place_tail = [&](bool transposed, int i, int64_t left, int64_t ld, int& s) -> int64_t {
        const int64_t k0 = static_cast<int64_t>(ktiles - 1) * BK;
        if (transposed) {
            const int64_t k = k0 + line_of(i), at = (k < K ? k : K - 1) * ld + first_row(i, left), last = (K - 1) * ld + left - 8;
            const int back = at > last ? static_cast<int>(at - last) : 0;
            s = k < K ? back : 8;
            return at - back;
        }
        const int64_t k = k0 + first_k(i);
        s = k > K - 8 ? static_cast<int>(k - (K - 8)) : 0;
        return (row_of(i) < left ? row_of(i) : left - 1) * ld + (k - s);
    };

    struct Regs {
        uint4 w[J], x[J];
    };
    Regs regs[2];   // tiles i and i + 1 of this split, the one that needs care being number 0
    int64_t off_w[J], off_x[J];
    int drop_w[J], drop_x[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int i = NW * j + wave;
        off_w[j] = place(WT, i, N - n0, p.ldw), off_x[j] = place(XT, i, M - m0, p.ldx);
        const int64_t tail_w = place_tail(WT, i, N - n0, p.ldw, drop_w[j]), tail_x = place_tail(XT, i, M - m0, p.ldx, drop_x[j]);
        if (full_tiles == 0) off_w[j] = tail_w, off_x[j] = tail_x;   // k-tile 0 is the one to be careful with
        const int64_t first = n > 0 ? t_begin : 0;
        regs[0].w[j] = load16(base_w + (has_tail ? tail_w : off_w[j] + first * step_w));
        regs[0].x[j] = load16(base_x + (has_tail ? tail_x : off_x[j] + first * step_x));
    }
    // Tile i >= 1; past the last one k-tile 0 again, which nobody multiplies.
    auto load = [&](int i, Regs& r) {
        const int t = i < n ? t_begin + i - has_tail : 0;
        const uint16_t *bw = base_w + t * step_w, *bx = base_x + t * step_x;
#pragma unroll
        for (int j = 0; j < J; ++j) r.w[j] = load16(bw + off_w[j]);
#pragma unroll
        for (int j = 0; j < J; ++j) r.x[j] = load16(bx + off_x[j]);
    };
    auto stash = [&](int slot, const Regs& r, int piece) {   // pieces 0 .. J - 1 are w's
        char* const to = lds + slot * kStage + (piece < J ? 0 : kX) + (NW * (piece % J) + wave) * 1024 + lane * 16;
        *reinterpret_cast<uint4*>(to) = piece < J ? r.w[piece % J] : r.x[piece % J];
    };
    load(1, regs[1]);
    if (has_tail) {
#pragma unroll
        for (int j = 0; j < J; ++j) regs[0].w[j] = drop(regs[0].w[j], drop_w[j]), regs[0].x[j] = drop(regs[0].x[j], drop_x[j]);
    }
#pragma unroll
    for (int q = 0; q < 2 * J; ++q) stash(0, regs[0], q);

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
    // The tile in `slot`: all fragments, the MFMAs of the first half, those of the second with between(q) in front of every
    // second one (q = 0 .. TN TM / 2 - 1).  The barriers to the scheduler keep that order.
    auto multiply = [&](int slot, auto between) {
        const char* const wt = lds + slot * kStage;
        bf16x8 fw[2][TN], fx[2][TM];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int a = 0; a < TN; ++a) fw[ks][a] = fragment(std::integral_constant<bool, WT>{}, wt, sub_w + a, ks);
#pragma unroll
            for (int b = 0; b < TM; ++b) fx[ks][b] = fragment(std::integral_constant<bool, XT>{}, wt + kX, sub_x + b, ks);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) acc[a][b] = mfma<F16>(fw[0][a], fx[0][b], acc[a][b]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) {
                if (b % 2 == 0) {
                    between((a * TM + b) / 2);
                    __builtin_amdgcn_sched_barrier(0);
                }
                acc[a][b] = mfma<F16>(fw[1][a], fx[1][b], acc[a][b]);
            }
    };
    constexpr int kPer = 2 * J / (TN * TM / 2);   // pieces written in front of each of them
    int i = 0;
#pragma unroll 1
    for (; i + 2 <= n; i += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            __syncthreads();   // tile i + u is complete; nobody reads the other slot any more
            load(i + u + 2, regs[u]);
            __builtin_amdgcn_sched_barrier(0);
            multiply(u, [&](int q) {
#pragma unroll
                for (int v = 0; v < kPer; ++v) stash(u ^ 1, regs[u ^ 1], q * kPer + v);
            });
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (i < n) {
        __syncthreads();
        multiply(0, [](int) {});
    }
    if (splits > 1) {   // lane order, so that the partial sums are written and read in whole lines
        floatx4* dst = reinterpret_cast<floatx4*>(partial) + (static_cast<int64_t>(block) * NW + wave) * (TN * TM * 64) + lane;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) dst[(a * TM + b) * 64] = acc[a][b];
        return;
    }
    // Through LDS, so that whole row segments of the tile leave 16 bytes a lane, at any address: with eight bytes a lane, as a
    // wavefront holds them, the adjoint of M 23, N 6400, K 2496 took 32.8 us, here 30.6.
    constexpr int kPitch = 2 * B + 16;   // staggers consecutive rows over the banks
    static_assert(B * kPitch <= 2 * kStage, "the result does not fit where the operands were");
    __syncthreads();   // nobody reads the operands any more
#pragma unroll
    for (int a = 0; a < TN; ++a) {
        const int64_t c = n0 + (sub_w + a) * 16 + 4 * kg;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < N) bv[e] = elem_to_f32<F16>(p.bias[c + e]);
        }
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f32_to_elem<F16>(acc[a][b][e] + bv[e]);
            *reinterpret_cast<uint2*>(lds + ((sub_x + b) * 16 + l16) * kPitch + ((sub_w + a) * 16 + 4 * kg) * 2) = make_uint2(o[0] | o[1] << 16, o[2] | o[3] << 16);
        }
    }
    __syncthreads();
    constexpr int kChunks = B / 8;   // of a row
#pragma unroll
    for (int q = 0; q < B * kChunks / kAnyThreads; ++q) {
        const int at = q * kAnyThreads + threadIdx.x, row = at / kChunks, chunk = at % kChunks;
        const int64_t m = m0 + row, c = n0 + chunk * 8;
        if (m >= M || c >= N) continue;
        const uint4 v = *reinterpret_cast<const uint4*>(lds + row * kPitch + chunk * 16);
        uint16_t* const dst = p.y + m * p.ldy + c;
        if (c + 8 <= N) {
            typedef u32x4 any __attribute__((aligned(2)));
            *reinterpret_cast<any*>(dst) = u32x4{v.x, v.y, v.z, v.w};
        } else {
            const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (c + e < N) dst[e] = static_cast<uint16_t>(words[e >> 1] >> (16 * (e & 1)));
        }
    }
}

// Two workgroups of 128 x 128 tiles share a CU (64 KiB of LDS and 256 registers each), four of 64 x 64.
template <bool F16, bool XT, bool WT, int T>
__global__ __launch_bounds__(kAnyThreads, T == 2 ? 2 : 4) void gemm16_any(const Part16 p, int splits, float* __restrict__ partial) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    any_product<F16, XT, WT, T>(p, blockIdx.x, splits, partial, lds);
}

// The adjoint of a linear shard in one launch: dx = dy . w and dw = dy^T . x by tiles of 64 TX and 64 TW, db = column sums of dy.
struct Adjoint16 {
    Part16 dx, dw;
    int splits_x, splits_w, blocks_x, blocks_w;   // workgroups of the products; of the sums of their splits
    int first_w;                                  // dw's workgroups come first
    float *partial_x, *partial_w;
    const uint16_t* dy;
    int64_t rows, cols, lddy;
    void* db;
    int strips;
};

template <bool F16, int TX, int TW>
__global__ __launch_bounds__(kAnyThreads, TX == 2 || TW == 2 ? 2 : 4) void linear16_adjoint(const Adjoint16 p) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    // Few strips of column sums come first, each a long chain of loads; many would keep the products waiting.
    const int products = p.blocks_x + p.blocks_w, first = p.strips <= kFirstStrips ? p.strips : 0;
    const int b = static_cast<int>(blockIdx.x) - first, x = p.first_w ? b - p.blocks_w : b, w = p.first_w ? b : b - p.blocks_x;
    if (b < 0 || b >= products) {
        typedef typename Elem<F16 ? 1 : 0>::type T;
        colsum_strip<F16 ? 1 : 0, kAnyThreads, 4>(reinterpret_cast<const T*>(p.dy), p.rows, p.cols, p.lddy, static_cast<T*>(p.db), b < 0 ? blockIdx.x : b - products,
                                                   p.strips, lds);
    } else if (x >= 0 && x < p.blocks_x) {
        any_product<F16, false, true, TX>(p.dx, x, p.splits_x, p.partial_x, lds);
    } else {
        any_product<F16, true, true, TW>(p.dw, w, p.splits_w, p.partial_w, lds);
    }
}

// The sums of the splits of both products; a product in one piece has no workgroups.
template <bool F16, int TX, int TW>
__global__ __launch_bounds__(256) void linear16_adjoint_sum(const Adjoint16 p, int blocks_x) {
    const int b = blockIdx.x;
    if (b < blocks_x) sum_splits<F16, 2, 2, 2 * TX, 2 * TX>(p.dx, p.splits_x, p.partial_x, b);
    else sum_splits<F16, 2, 2, 2 * TW, 2 * TW>(p.dw, p.splits_w, p.partial_w, b - blocks_x);
}

template <bool F16, int TX, int TW>
int launch_adjoint(const Adjoint16& p, hipStream_t s) {
    constexpr int lds_bytes = 4 * 64 * (TX > TW ? TX : TW) * kRowBytes;
    static_assert(colsum_lds_bytes(0, kAnyThreads) <= lds_bytes, "the column sums do not fit");
    hipLaunchKernelGGL((linear16_adjoint<F16, TX, TW>), dim3(static_cast<uint32_t>(p.blocks_x + p.blocks_w + p.strips)), dim3(kAnyThreads), lds_bytes, s, p);
    if (int rc = check_launch("linear16_adjoint")) return rc;
    const int sum_x = p.splits_x > 1 ? p.blocks_x / p.splits_x * 4 * TX * TX : 0, sum_w = p.splits_w > 1 ? p.blocks_w / p.splits_w * 4 * TW * TW : 0;
    if (sum_x + sum_w == 0) return 0;
    hipLaunchKernelGGL((linear16_adjoint_sum<F16, TX, TW>), dim3(static_cast<uint32_t>(sum_x + sum_w)), dim3(256), 0, s, p, sum_x);
    return check_launch("linear16_adjoint_sum");
}

template <bool F16>
__global__ __launch_bounds__(kAnyThreads) void gemm16_thin(const Part16 p, int64_t x_row, int64_t x_k, int64_t w_row, int64_t w_k, int64_t strips) {
    const int64_t m = blockIdx.x / strips, n = (blockIdx.x - m * strips) * kAnyThreads + threadIdx.x;
    if (n >= p.N) return;
    float v = 0.f;
    for (int64_t k = 0; k < p.K; ++k) v = fmaf(elem_to_f32<F16>(p.x[m * x_row + k * x_k]), elem_to_f32<F16>(p.w[n * w_row + k * w_k]), v);
    if (p.bias) v += elem_to_f32<F16>(p.bias[n]);
    p.y[m * p.ldy + n] = f32_to_elem<F16>(v);
}

template <bool F16, bool XT, bool WT, int T>
int launch_tiles(Part16 part, int splits, float* partial, hipStream_t s) {
    part.tiles_m = static_cast<int>((part.M + 64 * T - 1) / (64 * T)), part.tiles_n = static_cast<int>((part.N + 64 * T - 1) / (64 * T));
    const int ntiles = part.tiles_m * part.tiles_n;
    hipLaunchKernelGGL((gemm16_any<F16, XT, WT, T>), dim3(static_cast<uint32_t>(ntiles * splits)), dim3(kAnyThreads), 4 * 64 * T * kRowBytes, s, part,
                       splits, partial);
    if (int rc = check_launch("gemm16_any")) return rc;
    if (splits == 1) return 0;
    hipLaunchKernelGGL((gemm16_small_sum<F16, 2, 2, 2 * T, 2 * T>), dim3(static_cast<uint32_t>(ntiles * 4 * T * T)), dim3(256), 0, s, part, splits,
                       static_cast<const float*>(partial));
    return check_launch("gemm16_small_sum");
}

template <bool F16, bool XT, bool WT>
int launch_edge(const Small16& plan, const Part16& part, float* partial, hipStream_t s) {
    return plan.edge == 2 ? launch_tiles<F16, XT, WT, 2>(part, plan.splits, partial, s) : launch_tiles<F16, XT, WT, 1>(part, plan.splits, partial, s);
}

template <bool F16>
int launch(const Small16& plan, bool xt, bool wt, const Part16& part, float* partial, hipStream_t s) {
    if (plan.kind == Small16::kThin) {
        const int64_t strips = (part.N + kAnyThreads - 1) / kAnyThreads;
        hipLaunchKernelGGL((gemm16_thin<F16>), dim3(static_cast<uint32_t>(part.M * strips)), dim3(kAnyThreads), 0, s, part, xt ? 1 : part.ldx,
                           xt ? part.ldx : 1, wt ? 1 : part.ldw, wt ? part.ldw : 1, strips);
        return check_launch("gemm16_thin");
    }
    if (xt && wt) return launch_edge<F16, true, true>(plan, part, partial, s);
    if (xt) return launch_edge<F16, true, false>(plan, part, partial, s);
    if (wt) return launch_edge<F16, false, true>(plan, part, partial, s);
    return launch_edge<F16, false, false>(plan, part, partial, s);
}

}  // namespace

// Fits of a sweep over M 16 .. 8192, N 16 .. 12000, K 32 .. 8192 in the three layouts of a training step (28 000 products,
// 11 % off in the mean, picks 2.5 % behind the best of all ways measured), microseconds:
//   64 x 64    4.1 + 0.25 per k-tile and workgroup of a CU + 0.85 for every workgroup of a CU beyond the first; 8 % more where
//              not all are resident
//   128 x 128  6.1 + 0.62 and 2.5; 17 % more
//   splits     2.5 for the second launch and 3 for what it costs the host + the partial tiles, written and read, at 8 TB/s
//   at least   3 + operands and result once at 6 TB/s
// A CU works through whole workgroups while all are resident (four of 64 x 64, two of 128 x 128), else they even out.
// The other way -- operands copied into padded or transposed temporaries -- is 12 us of launches in front of the product plus
// the copies at 4.5 TB/s.  Measured among other steps, copies and product -> here: y of M 7001, N 1027, K 1001 42.4 -> 32.5 us,
// M 8191, N 1001, K 2051 59.0 -> 54.0; M 6001, N 1501, K 3001 71.7, here 105; M 4097, N 2049, K 2049 61, here 80.
Small16 plan_any16(bool xt, bool wt, int64_t M, int64_t N, int64_t K, int cus, int64_t workspace, double large_us) {
    Small16 best;
    double best_us = 12 + large_us + (static_cast<double>(M) + N) * K * 4 / 4.5e6;
    if (K < 8 && !(xt && wt)) {
        const int64_t strips = (N + kAnyThreads - 1) / kAnyThreads;
        if (strips <= 0xFFFFFF / M && 3 + static_cast<double>(M) * N / 2e6 < best_us) best.kind = Small16::kThin;
        return best;
    }
    const int64_t ktiles = (K + BK - 1) / BK;
    const double once_us = 3 + ((static_cast<double>(M) + N) * K + static_cast<double>(M) * N) * 2 / 6e6;
    for (const int edge : {1, 2}) {
        const int64_t tiles = ((M + 64 * edge - 1) / (64 * edge)) * ((N + 64 * edge - 1) / (64 * edge));
        const int64_t resident = edge == 1 ? 4 : 2, floats = edge * edge * 4096;
        if (tiles > 16 * static_cast<int64_t>(cus)) continue;
        for (const int splits : {1, 2, 3, 4, 6, 8, 12, 16}) {
            const int64_t workgroups = tiles * splits;
            if (splits > 1 && (workgroups > resident * cus || ktiles < 2 * splits || workgroups * floats > workspace)) break;
            const int64_t per_cu = (workgroups + cus - 1) / cus, steps = (ktiles + splits - 1) / splits;
            const double even = static_cast<double>(workgroups) / cus + 0.5;
            const double load = per_cu <= resident ? per_cu : even > resident ? even : resident;
            double us = edge == 1 ? 4.1 + steps * 0.25 * load + 0.85 * (load - 1) : 6.1 + steps * 0.62 * load + 2.5 * (load - 1);
            if (load > resident) us *= edge == 1 ? 1.08 : 1.17;
            if (us < once_us) us = once_us;
            if (splits > 1) us += 5.5 + static_cast<double>(workgroups) * floats * 8 / 8e6;
            if (us >= best_us) continue;
            best_us = best.us = us;
            best.kind = Small16::kAny, best.edge = edge, best.splits = splits, best.workspace = splits > 1 ? workgroups * floats : 0;
        }
    }
    return best;
}

// Both products on one chip at the same time: a workgroup's k-tile takes what it does above, the rounds of all of them are
// shared by the CUs, and the longest one is the least it can take; 4.1 or 6.1 as above, 5.5 for the launch that adds splits.
// The other way is `apart_us` for the products and 4.5 for the column sum, and 3 for each of the two further launches, of
// which 2 are the host's, where that may be what a step waits for.
// The best of these is taken if it also holds against what they leave out (careful_us): a long reduction in one piece takes 1.55
// times as long where rows are not aligned, and where it is by far the longest it waits for the other product's workgroups while
// not all are resident; the column sums take up to 2 ns a row; large products one after the other take 1.15 times `apart_us`.
// Three launches and one, of calls that therefore stay with three: M 5848, N 24, K 1408 aligned 22.9 and 29.6 us, M 8983, N 47,
// K 1624 39.6 and 62.1, M 8572, N 137, K 827 39.9 and 69.6, M 9975, N 17, K 37 19.6 and 28.2.  GPU time of 2204 calls for which
// the first estimate is for one launch (M 16 .. 16384, N 8 .. 8192, K 32 .. 8192, half of them aligned), in a replayed graph, which
// leaves out the host's share: 2069 take it, 1.5 times as fast as the three, 42 of them less than 0.95 times and at worst
// 0.79 (the former rule: 140 and 0.57); 12 of the 135 others would be faster by more than 5 % in one launch, at most 1.14 times.
// Of 1504 more calls with M above 2000, N up to 1024, drawn after the rule was made: 1312 take it, 1.3 times as fast, 75 less than 0.95
// times and at worst 0.62 (M 2146, N 19, K 931: 12.8 and 20.5 us; the former rule: 206 and 0.57), 24 of 192 lose, at most 1.24 times.
AdjointPlan16 plan_adjoint16(int64_t M, int64_t N, int64_t K, bool aligned, bool want_db, int cus, int64_t workspace, double apart_us) {
    AdjointPlan16 best;
    // operands along their rows have at least eight, dy read along n as well
    if (M < 8 || N < 8 || K < 8 || (want_db && M > kAdjointRows)) return best;
    const double launch_us = apart_us < 35 ? 3 : 1;
    const double other_us = apart_us + (want_db ? 4.5 + launch_us : 0) + launch_us;
    const int64_t strips = want_db ? (N + kNarrow - 1) / kNarrow : 0;
    double best_us = other_us, careful_us = 0;
    double least_us = 3 + 2 * (static_cast<double>(M) * N + (static_cast<double>(M) + N) * K * 2) / 6e6;   // operands and results once
    if (want_db && 4 + M * 0.0016 > least_us) least_us = 4 + M * 0.0016;                                       // one strip of the column sums
    for (int edges = 0; edges < 4; ++edges) {
        const int64_t ex = 1 + (edges & 1), ew = 1 + (edges >> 1);
        auto tiles = [](int64_t rows, int64_t cols, int64_t e) { return ((rows + 64 * e - 1) / (64 * e)) * ((cols + 64 * e - 1) / (64 * e)); };
        const int64_t tiles_x = tiles(M, K, ex), tiles_w = tiles(N, K, ew), kx = (N + BK - 1) / BK, kw = (M + BK - 1) / BK;
        const int64_t resident = (ex == 1 && ew == 1 ? 4 : 2) * static_cast<int64_t>(cus);
        if (tiles_x + tiles_w > 16 * static_cast<int64_t>(cus)) continue;
        const double cx = ex == 1 ? 0.25 : 0.62, cw = ew == 1 ? 0.25 : 0.62;
        for (const int sx : {1, 2, 3, 4, 6, 8}) {
            if (sx > 1 && (tiles_x * sx > resident || kx < 2 * sx)) break;
            for (const int sw : {1, 2, 3, 4, 6, 8}) {
                const int64_t bx = tiles_x * sx, bw = tiles_w * sw;
                const int64_t floats = (sx > 1 ? bx * ex * ex : 0) * 4096 + (sw > 1 ? bw * ew * ew : 0) * 4096;
                if ((sw > 1 && (bx + bw > resident || kw < 2 * sw)) || floats > workspace) break;
                const double nx = static_cast<double>((kx + sx - 1) / sx), nw = static_cast<double>((kw + sw - 1) / sw);
                const double all_x = bx * (nx * cx + (ex == 1 ? 0.85 : 2.5)) / cus, all_w = bw * (nw * cw + (ew == 1 ? 0.85 : 2.5)) / cus;
                const double all = (all_x + all_w) * 1.15, longest = nx * cx > nw * cw ? nx * cx : nw * cw;
                const double start_us = (ex == 1 && ew == 1 ? 4.1 : 6.1) + static_cast<double>(strips) / cus;
                const double sums_us = floats ? 5.5 + static_cast<double>(floats) * 8 / 8e6 : 0;
                double us = start_us + (all > longest ? all : longest);
                us = (us > least_us ? us : least_us) + sums_us;
                if (us >= best_us) continue;
                best_us = careful_us = us;
                best.edge_x = static_cast<int>(ex), best.edge_w = static_cast<int>(ew), best.splits_x = sx, best.splits_w = sw, best.workspace = floats;
                best.first_w = nw * cw > nx * cx;
                double chain = longest * (aligned ? 1 : 1.55);
                if (bx + bw > resident && chain > 1.5 * (all_x + all_w)) chain += 0.75 * (best.first_w ? all_x : all_w);
                for (const double t : {start_us + chain, want_db ? 4 + M * 0.002 : 0}) careful_us = t + sums_us > careful_us ? t + sums_us : careful_us;
            }
        }
    }
    return careful_us < (apart_us < 35 ? 1 : 1.15) * other_us ? best : AdjointPlan16{};
}

int run_adjoint16(const AdjointPlan16& plan, bool f16, const Part16& dx, const Part16& dw, void* db, float* workspace, hipStream_t s) {
    Adjoint16 p{};
    p.dx = dx, p.dw = dw, p.splits_x = plan.splits_x, p.splits_w = plan.splits_w, p.first_w = plan.first_w;
    auto tile = [](Part16& part, int edge) {
        part.tiles_m = static_cast<int>((part.M + 64 * edge - 1) / (64 * edge)), part.tiles_n = static_cast<int>((part.N + 64 * edge - 1) / (64 * edge));
        return part.tiles_m * part.tiles_n;
    };
    p.blocks_x = tile(p.dx, plan.edge_x) * plan.splits_x, p.blocks_w = tile(p.dw, plan.edge_w) * plan.splits_w;
    p.partial_x = workspace, p.partial_w = workspace + (plan.splits_x > 1 ? static_cast<int64_t>(p.blocks_x) * plan.edge_x * plan.edge_x * 4096 : 0);
    p.dy = dx.x, p.rows = dx.M, p.cols = dx.K, p.lddy = dx.ldx, p.db = db;
    p.strips = db ? static_cast<int>((p.cols + kNarrow - 1) / kNarrow) : 0;
    const int kind = (f16 ? 4 : 0) + (plan.edge_x == 2 ? 2 : 0) + (plan.edge_w == 2 ? 1 : 0);
    switch (kind) {
        case 0: return launch_adjoint<false, 1, 1>(p, s);
        case 1: return launch_adjoint<false, 1, 2>(p, s);
        case 2: return launch_adjoint<false, 2, 1>(p, s);
        case 3: return launch_adjoint<false, 2, 2>(p, s);
        case 4: return launch_adjoint<true, 1, 1>(p, s);
        case 5: return launch_adjoint<true, 1, 2>(p, s);
        case 6: return launch_adjoint<true, 2, 1>(p, s);
        default: return launch_adjoint<true, 2, 2>(p, s);
    }
}

int run_any16(const Small16& plan, bool f16, bool xt, bool wt, const Part16& part, float* partial, hipStream_t s) {
    return f16 ? launch<true>(plan, xt, wt, part, partial, s) : launch<false>(plan, xt, wt, part, partial, s);
}

}  // namespace ddl
