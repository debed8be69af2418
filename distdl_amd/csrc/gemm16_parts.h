// Device code that the kernels for smaller 16-bit products share: one MFMA of
// either type, the store of a lane's four columns, the sum of a split reduction's
// partial tiles.
#ifndef DDL_GEMM16_PARTS_H
#define DDL_GEMM16_PARTS_H
#include "gemm16_small.h"

namespace ddl {
namespace {

template <bool F16>
__device__ inline floatx4 mfma(const bf16x8& a, const bf16x8& b, const floatx4& c) {
    if (F16) {
        typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
        f16x8 ha, hb;
        __builtin_memcpy(&ha, &a, 16);
        __builtin_memcpy(&hb, &b, 16);
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(ha, hb, c, 0, 0, 0);
    }
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Four consecutive columns n .. n + 3 of output row m.
template <bool F16>
__device__ inline void store_four(uint16_t* __restrict__ y, int64_t ldy, int64_t m, int64_t n, int64_t N, const float* v) {
    uint16_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f32_to_elem<F16>(v[e]);
    uint16_t* dst = y + m * ldy + n;
    if (n + 3 < N) {   // global memory takes the eight bytes at any alignment
        typedef uint32_t words __attribute__((ext_vector_type(2)));
        typedef words any __attribute__((aligned(2)));
        words pk;
        pk[0] = static_cast<uint32_t>(o[0]) | (static_cast<uint32_t>(o[1]) << 16);
        pk[1] = static_cast<uint32_t>(o[2]) | (static_cast<uint32_t>(o[3]) << 16);
        *reinterpret_cast<any*>(dst) = pk;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) dst[e] = o[e];
    }
}

// Sum of the splits' partial tiles, bias, rounding, by workgroup `workgroup` of 256 threads: a thread per lane register quartet of
// the product kernel.
template <bool F16, int NWM, int NWN, int TM, int TN>
__device__ inline void sum_splits(const Part16& p, int splits, const float* __restrict__ partial, int workgroup) {
    constexpr int BM = 16 * NWM * TM, BN = 16 * NWN * TN, kQuartets = BM * BN / 4;
    const int ntiles = p.tiles_m * p.tiles_n;
    constexpr int kBlocks = kQuartets / 256;
    static_assert(kBlocks * 256 == kQuartets, "tile does not split into workgroups");
    const int tile = workgroup / kBlocks;
    const int q = (workgroup - tile * kBlocks) * 256 + threadIdx.x;
    int tm, tn;
    tile_of_workgroup(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int lane = q & 63, block = (q >> 6) % (TN * TM), wave = (q >> 6) / (TN * TM);
    const int64_t m = static_cast<int64_t>(tm) * BM + ((wave % NWM) * TM + block % TM) * 16 + (lane & 15);
    const int64_t n = static_cast<int64_t>(tn) * BN + ((wave / NWM) * TN + block / TM) * 16 + 4 * (lane >> 4);
    if (m >= p.M || n >= p.N) return;
    const floatx4* src = reinterpret_cast<const floatx4*>(partial) + static_cast<int64_t>(tile) * kQuartets + q;
    const int64_t stride = static_cast<int64_t>(ntiles) * kQuartets;
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
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = s[e] + (p.bias && n + e < p.N ? elem_to_f32<F16>(p.bias[n + e]) : 0.f);
    store_four<F16>(p.y, p.ldy, m, n, p.N, v);
}

template <bool F16, int NWM, int NWN, int TM, int TN>
__global__ __launch_bounds__(256) void gemm16_small_sum(const Part16 p, int splits, const float* __restrict__ partial) {
    sum_splits<F16, NWM, NWN, TM, TN>(p, splits, partial, blockIdx.x);
}

}  // namespace
}  // namespace ddl
#endif  // DDL_GEMM16_PARTS_H
