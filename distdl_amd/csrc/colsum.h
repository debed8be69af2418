// Column sums of a matrix of 16-bit or fp32 elements, in fp32: element types, and the
// sum of few rows by one workgroup per 16 columns.
#ifndef DDL_COLSUM_H
#define DDL_COLSUM_H
#include "ddl_common.h"

#include <hip/hip_fp16.h>

namespace ddl {

constexpr uint32_t kColsumXcds = 8;    // workgroups are dealt to the XCDs in turn
constexpr int kNarrow = 16;            // columns of a strip
constexpr int kFirstStrips = 64;       // so many strips go ahead of the products they share a launch with

namespace {

// 16 bytes at the alignment of an element, which global memory takes.
template <typename T>
__device__ inline uint4 load16(const T* p) {
    struct __attribute__((packed, aligned(sizeof(T)))) Any {
        uint32_t word[4];
    };
    const Any w = *reinterpret_cast<const Any*>(p);
    return make_uint4(w.word[0], w.word[1], w.word[2], w.word[3]);
}

__device__ inline float bf16_to_f32(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }

__device__ inline uint16_t f32_to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if (f != f) return 0x7FC0;
    u += 0x7FFFu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

// Element types of the column sum: 0 = bf16, 1 = fp16, 2 = fp32.
template <int DT>
struct Elem;
template <>
struct Elem<0> {
    typedef uint16_t type;
    static __device__ float load(const uint16_t* p) { return bf16_to_f32(*p); }
    static __device__ void store(uint16_t* p, float f) { *p = f32_to_bf16(f); }
    static __device__ void load8(const uint16_t* p, float (&v)[8]) {
        const uint4 q = load16(p);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = __uint_as_float(w[e] << 16);
            v[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
        }
    }
};
template <>
struct Elem<1> {
    typedef __half type;
    static __device__ float load(const __half* p) { return __half2float(*p); }
    static __device__ void store(__half* p, float f) { *p = __float2half_rn(f); }
    static __device__ void load8(const __half* p, float (&v)[8]) {
        const uint4 q = load16(p);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float2 f = __half22float2(*reinterpret_cast<const __half2*>(&w[e]));
            v[2 * e] = f.x;
            v[2 * e + 1] = f.y;
        }
    }
};
template <>
struct Elem<2> {
    typedef float type;
    static __device__ float load(const float* p) { return *p; }
    static __device__ void store(float* p, float f) { *p = f; }
    static __device__ void load8(const float* p, float (&v)[8]) {
        load4(p, *reinterpret_cast<float(*)[4]>(&v[0]));
        load4(p + 4, *reinterpret_cast<float(*)[4]>(&v[4]));
    }
    static __device__ void load4(const float* p, float (&v)[4]) {
        const uint4 q = load16(p);
        v[0] = __uint_as_float(q.x), v[1] = __uint_as_float(q.y), v[2] = __uint_as_float(q.z), v[3] = __uint_as_float(q.w);
    }
};

constexpr int colsum_lds_bytes(int dt, int block) {   // row groups x 17 floats, and their sums
    return (block / (kNarrow / (dt == 2 ? 4 : 8)) * (kNarrow + 1) + block) * 4;
}

// Strip `strip` of `strips` of the column sums: all rows, 16 / E lanes per row (E elements of 16 bytes each, at any
// address), LDS folds the row groups.  Two stages (partial sums, then theirs) are two
// launches and a workspace for what is a few microseconds of reading: [777, 333] fp32 5.0
// + 4.7 us, [1024, 4096] bf16 4.9 + 3.9 us.  Neighbouring strips go to one XCD, so that a
// 128-byte line they share comes from memory once and not for each of four L2 caches, and rows
// that are not aligned are read 16 bytes a lane like others: [1024, 4096] bf16 5.7 ->
// 3.8 us, [944, 16382] 22 -> 10.  ACC chains of sums per lane: with a quarter of the lanes, four of
// them are as short as one of the others.
template <int DT, int BLOCK, int ACC>
__device__ inline void colsum_strip(const typename Elem<DT>::type* __restrict__ a, int64_t rows, int64_t cols, int64_t ld,
                                    typename Elem<DT>::type* __restrict__ out, uint32_t strip, uint32_t strips, char* lds) {
    typedef typename Elem<DT>::type T;
    constexpr int E = 16 / static_cast<int>(sizeof(T)), kPieces = kNarrow / E, kGroups = BLOCK / kPieces;
    float (*const fold)[kNarrow + 1] = reinterpret_cast<float (*)[kNarrow + 1]>(lds);
    float (*const half)[kNarrow] = reinterpret_cast<float (*)[kNarrow]>(lds + kGroups * (kNarrow + 1) * 4);
    const int t = threadIdx.x, g = t / kPieces, c = t % kPieces * E;
    const uint32_t per = strips / kColsumXcds, whole = per * kColsumXcds;   // hardware deals workgroups round-robin over the XCDs
    const int64_t c0 = static_cast<int64_t>(strip < whole ? strip % kColsumXcds * per + strip / kColsumXcds : strip) * kNarrow;
    const int64_t gc = c0 + c;
    float acc[ACC][E];
#pragma unroll
    for (int u = 0; u < ACC; ++u)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[u][e] = 0.f;
    // The last vector of a row ends with it: its first `back` columns are the vector's before it, added there.
    const int back = gc + E > cols ? static_cast<int>(gc + E - cols) : 0;
    if (back < E && gc >= back) {
        const T* const first = a + (gc - back);
        auto add = [&](int64_t r, float (&to)[E]) {
            float v[E];
            if constexpr (sizeof(T) == 2) Elem<DT>::load8(first + r * ld, v);
            else Elem<DT>::load4(first + r * ld, v);
#pragma unroll
            for (int e = 0; e < E; ++e) to[e] += v[e];
        };
        int64_t r = g;
        if constexpr (ACC > 1) {
            for (; r + (ACC - 1) * kGroups < rows; r += ACC * kGroups)
#pragma unroll
                for (int u = 0; u < ACC; ++u) add(r + u * kGroups, acc[u]);
        }
#pragma unroll 4
        for (; r < rows; r += kGroups) add(r, acc[0]);
#pragma unroll
        for (int d = ACC / 2; d > 0; d /= 2)
#pragma unroll
            for (int u = 0; u < d; ++u)
#pragma unroll
                for (int e = 0; e < E; ++e) acc[u][e] += acc[u + d][e];
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (e >= back) fold[g][c + e - back] = acc[0][e];
    } else if (back < E) {   // rows shorter than a vector
        for (int64_t r = g; r < rows; r += kGroups)
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (gc + e < cols) acc[0][e] += Elem<DT>::load(a + r * ld + gc + e);
#pragma unroll
        for (int e = 0; e < E; ++e) fold[g][c + e] = acc[0][e];
    }
    __syncthreads();
    constexpr int kParts = BLOCK / kNarrow;   // threads per column
    const int col = t % kNarrow, part = t / kNarrow;
    // Sums of many partial sums go pairwise: added one after the other, 64 of them lose a third more to rounding in fp32 than
    // the two stages do.
    constexpr int kMine = kGroups / kParts;
    float mine[kMine];
#pragma unroll
    for (int k = 0; k < kMine; ++k) mine[k] = fold[part + k * kParts][col];
#pragma unroll
    for (int d = kMine / 2; d > 0; d /= 2)
#pragma unroll
        for (int k = 0; k < d; ++k) mine[k] += mine[k + d];
    half[part][col] = mine[0];
    __syncthreads();
    if (t < kNarrow && c0 + t < cols) {
        float r[kParts];
#pragma unroll
        for (int k = 0; k < kParts; ++k) r[k] = half[k][t];
#pragma unroll
        for (int d = kParts / 2; d > 0; d /= 2)
#pragma unroll
            for (int k = 0; k < d; ++k) r[k] += r[k + d];
        Elem<DT>::store(out + c0 + t, r[0]);
    }
}

}  // namespace
}  // namespace ddl
#endif  // DDL_COLSUM_H
