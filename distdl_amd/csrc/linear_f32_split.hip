// fp32 linear products on the bf16 matrix cores, without loss:
// y[M,N] = a[M,K] . b[N,K]^T + bias[N], fp32 in and out.
//
// An fp32 value is the sum of three bf16 values, exactly: its rounding to bf16, the
// rounding of what is left, and what is left then (8 + 8 + 8 significant bits), as
// published by Henry, Tang and Heinecke ("Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", 2019).  Elements are
// multiplied by 2^24 first: then no part of any of them, denormal ones included, is
// below bf16's normal range.  Of the nine products of two such sums the smallest is
// below 2^-33 of the product and left out; the other eight go through
// v_mfma_f32_32x32x16_bf16, which accumulates in fp32: 256 cycles for 32 x 32 x 16 where
// v_mfma_f32_32x32x2_f32 takes 512.
//
// The products of the first parts have an accumulator of their own; they are rounded
// once per 16 terms, and a term that is zero rounds nothing.  The seven others, together
// below 2^-7 of them, have a second one, added once at the end.  (All in one accumulator
// round once per part-product at its full size: 0.5 to 1.5 times the fp32 instruction's
// error, the more the fewer terms are not zero.  With the six largest products alone a
// sum of one term is 1.025 times as far off.)  Error against float64 in the 2-norm,
// fp32 instruction -> here, M = N = 1408, K 8192, share of x that is not zero: all 1.62e-6 -> 0.40e-6, a quarter
// 0.81e-6 -> 0.23e-6, a hundredth 0.164e-6 -> 0.055e-6, one element a row 0.0253e-6 both.
//
// Bound by the matrix instructions' power and, in small products, by issue: while a CU's
// wavefronts multiply, they split (seven instructions an element).  149 to 160 TFLOP/s
// in large products, where the fp32 instruction ends at 148 (M 8192, N 3584, K 8192 3.06 to
// 3.10 ms, its adjoint 3.10 and 3.22).  Measured, fp32 instruction (64 x 64 or
// 256 x 256 tiles) -> here, operands along k or along their rows: M 256, N 3551, K 6575
// 116 -> 101 to 106 us, M 3551, N 6575, K 256 147 to 169 -> 99 to 105, M = N = K = 2048 140 -> 122
// to 128, 4096 968 -> 858 to 897, M 1024, N 8192, K 8192 1050 to 1075 -> 861 to 903; below about 20 us
// the smaller tiles are faster.
//
//   workgroup  256 threads = 4 wavefronts (2 x 2), tile 128 x 128 x 16(k); a wavefront
//              has 2 x 2 blocks of 32 x 32
//   global     a thread fetches eight k of a row of each operand into registers, three
//              k-tiles ahead: 32 bytes of the row, or eight rows' worth of dwords for
//              an operand contiguous along its rows.  Any pitch, length and
//              4-byte-aligned address
//   LDS        every element is split once per workgroup, on its way into LDS: three
//              planes of rows of 32 bytes, halves swapped in eight rows of sixteen, so
//              that 16 lanes reading one half of 16 rows, or writing it, meet no bank
//              twice.  Two stages
//   splits     workgroups share the reduction of a tile through a workspace, whose
//              sums gemm32_small_sum adds
//
// What the parts cannot carry is found on the way: every thread keeps the largest
// magnitude that it fetches.  Tiles with infinities, elements from 2^100 on, or
// elements whose product times the length of the reduction reaches 2^78 (which scaled
// might pass the largest float) are computed again from memory on
// v_mfma_f32_32x32x2_f32.
#include "gemm32_small.h"
#include "gemm_tiles.h"
#include <type_traits>

namespace ddl {
namespace {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr int kBlock = 256;
constexpr int kTile = 128, BK = 16;
constexpr int kAhead = 3;               // k-tiles in flight from memory
constexpr int kTurns = 2 * kAhead;      // k-tiles until both the registers and the two stages of LDS come round
constexpr int kRowSpan = 2 * BK;        // bytes of a row in a plane
constexpr int kPlane = kTile * kRowSpan, kOperand = 3 * kPlane, kStage = 2 * kOperand;   // a stage: the w planes, then the x planes
constexpr int kOutPitch = 68;           // floats of a row of results in LDS: 64 and room for 16 rows on 64 banks
constexpr float kScale = 0x1p24f, kUnscale = 0x1p-48f;   // of an element before it is split, of a result
constexpr float kHuge = 0x1p100f, kMost = 0x1p78f;       // what elements and sums may reach, unscaled

typedef PartOf<float> Part32;

// Two floats as two bf16 each in three planes.
__device__ inline void split2(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    auto rounded = [](float x, float y) {
        floatx2 v;
        v[0] = x, v[1] = y;
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    };
    hi = rounded(a, b);
    a -= __uint_as_float(hi << 16), b -= __uint_as_float(hi & 0xFFFF0000u);
    mid = rounded(a, b);
    a -= __uint_as_float(mid << 16), b -= __uint_as_float(mid & 0xFFFF0000u);
    lo = rounded(a, b);
}

// 16-byte chunk `octet` of a row in a plane.
__device__ inline int chunk_at(int row, int octet) { return row * kRowSpan + ((octet ^ ((row >> 3) & 1)) << 4); }

// One operand's part of a k-tile, 128 rows x 16 k: a thread has eight k of a row.
template <bool TRANSPOSED>
struct Fetch {
    const float* p;        // first of this thread's eight elements of the next k-tile
    int64_t ld;
    int row, octet;
    float most;            // largest magnitude fetched

    __device__ void init(const float* base, int64_t origin, int64_t rows, int64_t pitch, int64_t k0) {
        ld = pitch;
        const int t = threadIdx.x;
        // along k: two lanes share a row; along rows: lanes along the rows
        row = TRANSPOSED ? t % kTile : t / 2;
        octet = TRANSPOSED ? t / kTile : t % 2;
        most = 0.f;
        at(base, origin, rows, k0);
    }
    __device__ void at(const float* base, int64_t origin, int64_t rows, int64_t k0) {
        const int64_t r = origin + row < rows ? origin + row : rows - 1;   // rows past the end repeat the last one
        const int64_t k = k0 + 8 * octet;
        p = base + (TRANSPOSED ? k * ld + r : r * ld + k);
    }
    __device__ void load(float (&v)[8], bool forward) {   // then on to the next k-tile, if there is one
        typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
        if (TRANSPOSED) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = p[e * ld];
        } else {
            const quad a = *reinterpret_cast<const quad*>(p), b = *reinterpret_cast<const quad*>(p + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
        }
        p += forward ? (TRANSPOSED ? BK * ld : BK) : 0;
    }
    __device__ void load_last(float (&v)[8], int64_t left) {   // of the k-tile there are `left` < BK elements
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 8 * octet + e < left ? p[TRANSPOSED ? e * ld : e] : 0.f;
    }
    __device__ void store(const float (&v)[8], char* planes) {
        uint32_t w[3][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            most = fmaxf(fmaxf(most, fabsf(v[2 * e])), fabsf(v[2 * e + 1]));
            split2(v[2 * e] * kScale, v[2 * e + 1] * kScale, w[0][e], w[1][e], w[2][e]);
        }
        char* at = planes + chunk_at(row, octet);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            u32x4 q;
            q[0] = w[s][0], q[1] = w[s][1], q[2] = w[s][2], q[3] = w[s][3];
            *reinterpret_cast<u32x4*>(at + s * kPlane) = q;
        }
    }
};

template <bool XT, bool WT>
__global__ __launch_bounds__(kBlock, 2) void gemm32_split(const Part32 p, int splits, float* __restrict__ partial) {
    __shared__ __attribute__((aligned(16))) char lds[2 * kStage];
    const int ntiles = p.tiles_m * p.tiles_n;
    const int split = static_cast<int>(blockIdx.x) / ntiles, tile = static_cast<int>(blockIdx.x) - split * ntiles;
    int tm, tn;
    tile_of_workgroup(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int64_t M = p.M, N = p.N, K = p.K;
    const int64_t m0 = static_cast<int64_t>(tm) * kTile, n0 = static_cast<int64_t>(tn) * kTile;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, kh = lane >> 5;
    const int sub_w = (wave >> 1) * 2, sub_x = (wave & 1) * 2;   // first 32-row block of this wavefront in the w and x tiles
    const int64_t ktiles = (K + BK - 1) / BK, per = (ktiles + splits - 1) / splits;
    const int64_t t_begin = split * per < ktiles ? split * per : ktiles, t_end = t_begin + per < ktiles ? t_begin + per : ktiles;

    floatx16 acc[2][2], rest[2][2];   // [n block][m block]: the products of the first parts, and all others
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = rest[i][j][e] = 0.f;
    };
    clear();
    Fetch<WT> fw;
    Fetch<XT> fx;
    fw.init(p.w, n0, N, p.ldw, t_begin * BK);
    fx.init(p.x, m0, M, p.ldx, t_begin * BK);
    const int64_t full = t_end * BK <= K || t_begin == t_end ? t_end : t_end - 1;   // k-tiles up to here are whole
    // Elements k = 8 kh + {0..7} of row l32 of a block, of plane s.
    auto fragment = [&](const char* planes, int s, int block) {
        return *reinterpret_cast<const bf16x8*>(planes + s * kPlane + chunk_at(block * 32 + l32, kh));
    };
    auto multiply = [&](const char* at, auto&& between) {
        bf16x8 a[3][2], b[3][2];
        auto read = [&](int s) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[s][i] = fragment(at, s, sub_w + i);
                b[s][i] = fragment(at + kOperand, s, sub_x + i);
            }
        };
        auto term = [&](floatx16 (&to)[2][2], int sw, int sx) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[sw][i], b[sx][j], to[i][j], 0, 0, 0);
        };
        // Splitting and storing the next k-tile goes into the shadow of the matrix instructions, six at a time: left alone,
        // the compiler puts all of it in front of them (six part-products: 2048 x 2048 x 2048 107 us instead of 93).
        auto alternate = [](auto reads, auto products) {
            __builtin_amdgcn_sched_group_barrier(0x100, decltype(reads)::value, 0);    // LDS reads
#pragma unroll
            for (int i = 0; i < decltype(products)::value; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // a matrix instruction
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);   // others of the vector ALU
            }
        };
        // The third parts are read when twelve products are under way: all at once they would not fit the registers.
        read(0), read(1);
        between();
        term(acc, 0, 0), term(rest, 1, 1), term(rest, 1, 0), term(rest, 0, 1);
        read(2);
        term(rest, 2, 1), term(rest, 1, 2), term(rest, 2, 0), term(rest, 0, 2);
        alternate(std::integral_constant<int, 8>{}, std::integral_constant<int, 12>{});
        alternate(std::integral_constant<int, 4>{}, std::integral_constant<int, 20>{});
    };
    if (t_begin < full) {
        // The loads are never skipped (past the last whole k-tile that one is loaded again): with a branch around them the
        // compiler could not count which have landed and would wait for all.
        float vw[kAhead][8], vx[kAhead][8];
        int64_t next = t_begin;   // the k-tile that is loaded next
        auto load = [&](int i) {
            const bool forward = next + 1 < full;
            fw.load(vw[i], forward);
            fx.load(vx[i], forward);
            next += forward ? 1 : 0;
        };
#pragma unroll
        for (int i = 0; i < kAhead; ++i) load(i);
        fw.store(vw[0], lds);
        fx.store(vx[0], lds + kOperand);
        load(0);
        int64_t t = t_begin;
        while (true) {
#pragma unroll
            for (int i = 0; i < kTurns; ++i) {
                // This wavefront's part of k-tile t is in LDS and its reads of the other stage have returned; the loads stay in flight.
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                multiply(lds + (i & 1) * kStage, [&]() {
                    fw.store(vw[(i + 1) % kAhead], lds + ((i + 1) & 1) * kStage);
                    fx.store(vx[(i + 1) % kAhead], lds + ((i + 1) & 1) * kStage + kOperand);
                    load((i + 1) % kAhead);
                });
                if (++t == full) break;
            }
            if (t == full) break;
        }
        __syncthreads();
    }
    if (full < t_end) {
        fw.at(p.w, n0, N, full * BK);
        fx.at(p.x, m0, M, full * BK);
        float vw[8], vx[8];
        fw.load_last(vw, K - full * BK);
        fx.load_last(vx, K - full * BK);
        fw.store(vw, lds);
        fx.store(vx, lds + kOperand);
        __syncthreads();
        multiply(lds, [] {});
        __syncthreads();
    }

    // Largest magnitudes of the operands' parts of the tile.
    uint32_t* const largest = reinterpret_cast<uint32_t*>(lds);   // floats >= 0 compare like integers
    if (threadIdx.x < 2) largest[threadIdx.x] = 0;
    __syncthreads();
    atomicMax(&largest[0], __float_as_uint(fw.most));
    atomicMax(&largest[1], __float_as_uint(fx.most));
    __syncthreads();
    const float most_w = __uint_as_float(largest[0]), most_x = __uint_as_float(largest[1]);
    const bool odd = !(most_w < kHuge) || !(most_x < kHuge) || !(most_w * most_x * static_cast<float>((t_end - t_begin) * BK) < kMost);
    if (odd) {   // the same in all threads
        clear();
        auto element = [&](const float* base, bool transposed, int64_t row, int64_t rows, int64_t ld, int64_t k) {
            row = row < rows ? row : rows - 1;
            const bool inside = k < K;
            const float f = base[inside ? (transposed ? k * ld + row : row * ld + k) : 0];
            return inside ? f : 0.f;
        };
#pragma unroll 1
        for (int64_t k = t_begin * BK; k < t_end * BK; k += 2) {
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i] = element(p.w, WT, n0 + (sub_w + i) * 32 + l32, N, p.ldw, k + kh);
                b[i] = element(p.x, XT, m0 + (sub_x + i) * 32 + l32, M, p.ldx, k + kh);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }

    else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = (acc[i][j][e] + rest[i][j][e]) * kUnscale;
    }

    // Lane holds row m = l32 and columns n = 8 g + 4 kh + {0..3} of a block in acc[4 g + {0..3}].
    auto quad = [&](int i, int j, int g) { return floatx4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]}; };
    if (splits > 1) {   // block (m, n) of the tile is number m + 4 n, as gemm32_small_sum counts them
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int64_t block = static_cast<int64_t>(blockIdx.x) * 16 + sub_x + j + 4 * (sub_w + i);
                    reinterpret_cast<floatx4*>(partial)[block * 256 + g * 64 + lane] = quad(i, j, g);
                }
        return;
    }
    // Through LDS, 32 rows of 64 results of a wavefront at a time, so that sixteen lanes store a row of 256 bytes: with the
    // four floats a lane holds, rows that are no multiple of four went out a float at a time in pieces of 32 bytes (M 3551,
    // N 6575, K 256 133 us, here 84).
    __syncthreads();   // the largest magnitudes have been read
    float* const out = reinterpret_cast<float*>(lds) + wave * (32 * kOutPitch);
    const int64_t n = n0 + sub_w * 32 + (lane & 15) * 4;
    const floatx4 bias = bias_of(p.bias, n < N ? n : N - 1, N);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) *reinterpret_cast<floatx4*>(&out[l32 * kOutPitch + 32 * i + 8 * g + 4 * kh]) = quad(i, j, g);
        __builtin_amdgcn_wave_barrier();   // one wavefront writes and reads: LDS serves it in order
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int row = 4 * r + (lane >> 4);
            const floatx4 v = *reinterpret_cast<const floatx4*>(&out[row * kOutPitch + (lane & 15) * 4]) + bias;
            const int64_t m = m0 + (sub_x + j) * 32 + row;
            if (m >= M) continue;
            float* const dst = p.y + m * p.ldy + n;
            if (n + 3 < N) {
                typedef floatx4 any __attribute__((aligned(4)));
                *reinterpret_cast<any*>(dst) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) dst[e] = v[e];
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <bool XT, bool WT>
int launch(Part32 part, int splits, float* partial, hipStream_t s) {
    part.tiles_m = static_cast<int>((part.M + kTile - 1) / kTile), part.tiles_n = static_cast<int>((part.N + kTile - 1) / kTile);
    hipLaunchKernelGGL((gemm32_split<XT, WT>), dim3(static_cast<uint32_t>(part.tiles_m * part.tiles_n * splits)), dim3(kBlock), 0, s, part, splits, partial);
    if (int rc = check_launch("gemm32_split")) return rc;
    return splits == 1 ? 0 : sum_small32(part, 4, splits, partial, s);
}

}  // namespace

// The estimates are fits to a sweep over M, N, K of 64 .. 8192 on all operand layouts, in microseconds: 6 + for each tile that a
// CU has to work through 4.5 and, per 32 of its reduction, 1.57 (few CUs at work) to 1.72 (all) + for splits a second launch (2.3,
// and 5 for what it and the workspace cost the host) and the partial tiles at 5 TB/s.  Over 66 sizes in three layouts the way they
// choose is on average 1.1 % slower than the faster of both kernels and all splits.
Small32 plan_split32(int64_t M, int64_t N, int64_t K, int cus, int64_t workspace, const Small32& other) {
    Small32 best;
    const int64_t ktiles = (K + BK - 1) / BK, tiles = ((M + kTile - 1) / kTile) * ((N + kTile - 1) / kTile);
    if (tiles > 0xFFFFFF) return best;   // a launch has fewer than 2^32 threads, 256 per tile
    double best_us = other.groups ? other.us : 1e30;
    for (const int splits : {1, 2, 3, 4, 6, 8, 12, 16}) {
        if (splits > 1 && (tiles * splits > 4 * static_cast<int64_t>(cus) || ktiles < 8 * splits || tiles * splits * kTile * kTile > workspace)) break;
        // Fewer, longer sums than the other way are only taken where this kernel's smaller rounding error makes up for it (0.24 to
        // 0.34 of the other's for dense sums of the same length; it grows by their square root).
        if (4 * splits < other.groups * other.splits) continue;
        const int64_t all = tiles * splits, per_cu = (all + cus - 1) / cus, kt = (ktiles + splits - 1) / splits;
        const double fill = all < cus ? static_cast<double>(all) / cus : 1.0;
        double us = 6 + per_cu * (4.5 + 0.5 * static_cast<double>(kt) * (1.57 + 0.15 * fill));
        if (splits > 1) us += 7.3 + static_cast<double>(all) * kTile * kTile * 8 / 5e6;
        if (us >= best_us) continue;
        best_us = best.us = us;
        best.edge = kTile, best.splits = splits, best.workspace = splits > 1 ? all * kTile * kTile : 0;
    }
    return best;
}

int run_split32(const Small32& plan, bool xt, bool wt, const PartOf<float>& part, float* partial, hipStream_t s) {
    if (xt && wt) return launch<true, true>(part, plan.splits, partial, s);
    if (xt) return launch<true, false>(part, plan.splits, partial, s);
    if (wt) return launch<false, true>(part, plan.splits, partial, s);
    return launch<false, false>(part, plan.splits, partial, s);
}

}  // namespace ddl
