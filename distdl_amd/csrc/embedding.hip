// DistributedEmbedding shard gather (reference: nn/embedding.py:244-246,
// torch.nn.functional.embedding on the local table).  out[t] is row ids[t]-lo of
// the table when lo <= ids[t] < hi and a row of zero bits otherwise.  Rows are
// opaque bytes, moved 16 at a time.
//
// max_norm (the renormalisation F.embedding performs before the lookup): the
// rows that are looked up are flagged, then one wavefront per flagged row forms
// the p-norm in fp32 and, where it exceeds max_norm, scales the row in place by
// max_norm / (norm + 1e-7) -- once per row however often it is looked up.
#include "ddl_common.h"
#include "ln_elements.h"

namespace ddl {
namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr uint32_t kXcds = 8;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// How the rows are moved: as vectors of 16 bytes with streaming stores.  Bound by HBM, and
// for misses by how the stores of a moment lie in it; nothing is in a cache when a step gets
// here, so all was measured on tables, ids and outputs that change from call to call, with the
// adjoint behind each call.
//
// gather_rows: 256 lanes per row, which fill it or most of it, 4 KiB after 4 KiB; its id is a
// scalar.  131 072 ids into [16032, 4096] bf16, of which one in eight hits, 255 us with the
// adjoint (one wavefront per row, eight vectors in flight, 275; 512 lanes 286; 256 with two
// vectors each at a time 271; gather_vectors 279).
// gather_vectors: the vectors of the whole output in a row, two per lane of 512, for rows that
// 256 lanes do not fill: 60 000 ids into [16000, 3000], one in eight hits, 103 us (by rows 118,
// by wavefronts 127).
// ANY: rows or addresses that are no multiples of 16 bytes, any of them; the last vector
// of a row ends with it, and neighbouring workgroups run on one XCD, whose L2 puts the lines
// together that two of them write: 32 768 ids into [6155, 3895] bf16 114 -> 71 us, 8 416
// into [65590, 2863] 41 -> 18, 224 into [1944, 4051] fp32 10.6 -> 4.5 (before: a vector of
// an element's size per lane).
template <bool ANY>
__device__ inline u32x4 load_vector(const char* p) {
    typedef u32x4 any __attribute__((aligned(1)));
    return ANY ? *reinterpret_cast<const any*>(p) : *reinterpret_cast<const u32x4*>(p);
}
template <bool ANY>
__device__ inline void store_vector(char* p, u32x4 v) {
    typedef u32x4 any __attribute__((aligned(1)));
    if (ANY) __builtin_nontemporal_store(v, reinterpret_cast<any*>(p));
    else __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}
template <bool ANY>
__device__ inline uint32_t block_number() {   // hardware deals workgroups round-robin over the XCDs
    const uint32_t per = gridDim.x / kXcds, whole = per * kXcds;
    return ANY && blockIdx.x < whole ? blockIdx.x % kXcds * per + blockIdx.x / kXcds : blockIdx.x;
}

template <bool ANY, typename IdT>
__global__ __launch_bounds__(kBlock) void gather_rows(const char* __restrict__ weight, int64_t ldw_bytes, uint32_t nvec, int64_t last,
                                                      const IdT* __restrict__ ids, int64_t lo, int64_t hi, char* __restrict__ out, int64_t row_bytes) {
    const uint32_t t = block_number<ANY>();
    const int64_t id = static_cast<int64_t>(ids[t]);
    char* const dst = out + static_cast<int64_t>(t) * row_bytes;
    auto place = [&](uint32_t c) { return ANY && c + 1 == nvec ? last : static_cast<int64_t>(c) * 16; };
    if (id >= lo && id < hi) {
        const char* const src = weight + (id - lo) * ldw_bytes;
        for (uint32_t c = threadIdx.x; c < nvec; c += kBlock) store_vector<ANY>(dst + place(c), load_vector<ANY>(src + place(c)));
    } else {
        for (uint32_t c = threadIdx.x; c < nvec; c += kBlock) store_vector<ANY>(dst + place(c), u32x4{0, 0, 0, 0});
    }
}

constexpr int kGatherBlock = 512, kGatherVectors = 2;

template <bool ANY, typename IdT>
__global__ __launch_bounds__(kGatherBlock) void gather_vectors(const char* __restrict__ weight, int64_t ldw_bytes, uint32_t nvec, FastDiv by_nvec,
                                                               int64_t last, const IdT* __restrict__ ids, uint32_t total, int64_t lo, int64_t hi,
                                                               char* __restrict__ out, int64_t row_bytes) {
    const uint32_t first = block_number<ANY>() * (kGatherBlock * kGatherVectors) + threadIdx.x;
    u32x4 v[kGatherVectors];
    int64_t to[kGatherVectors];
#pragma unroll
    for (int u = 0; u < kGatherVectors; ++u) {
        const uint32_t i = first + u * kGatherBlock < total ? first + u * kGatherBlock : total - 1, t = fd_div(i, by_nvec), c = i - t * nvec;
        const int64_t id = static_cast<int64_t>(ids[t]);
        const int64_t at = ANY && c + 1 == nvec ? last : static_cast<int64_t>(c) * 16;
        to[u] = static_cast<int64_t>(t) * row_bytes + at;
        v[u] = u32x4{0, 0, 0, 0};
        if (id >= lo && id < hi) {   // misses issue no load
            v[u] = load_vector<ANY>(weight + (id - lo) * ldw_bytes + at);
        }
    }
#pragma unroll
    for (int u = 0; u < kGatherVectors; ++u)
        if (first + u * kGatherBlock < total) store_vector<ANY>(out + to[u], v[u]);
}

// Rows of less than 16 bytes: an element per lane.
template <typename V, typename IdT>
__global__ __launch_bounds__(kBlock) void gather_elements(const char* __restrict__ weight, int64_t ldw_bytes, uint32_t dim, FastDiv by_dim,
                                                          const IdT* __restrict__ ids, uint32_t total, int64_t lo, int64_t hi, V* __restrict__ out) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= total) return;
    const uint32_t t = fd_div(i, by_dim), c = i - t * dim;
    const int64_t id = static_cast<int64_t>(ids[t]);
    V v = 0;
    if (id >= lo && id < hi) v = reinterpret_cast<const V*>(weight + (id - lo) * ldw_bytes)[c];
    out[i] = v;
}

// Lanes are numbered in 31 bits, and a launch has fewer than 2^32 threads: slabs of as many ids as that takes.
template <typename IdT>
int launch_gather(const char* w, int64_t ldw_bytes, int64_t row_bytes, int64_t elem, const IdT* ids, int64_t n, int64_t lo, int64_t hi, char* out, hipStream_t s) {
    const bool vectors = row_bytes >= 16, any = ((row_bytes | ldw_bytes | reinterpret_cast<intptr_t>(w) | reinterpret_cast<intptr_t>(out)) & 15) != 0;
    const int64_t lanes = vectors ? (row_bytes + 15) / 16 : row_bytes / elem;
    const bool by_rows = vectors && lanes * 10 >= (lanes + kBlock - 1) / kBlock * kBlock * 9;
    const int64_t most = by_rows ? 0xFFFFFF : 0x7FFF0000ll / lanes;
    if (lanes > 0x7FFF0000ll) return fail(DDL_E_UNSUPP, "embedding gather: rows of %lld bytes", (long long)row_bytes);
    const FastDiv div = make_fastdiv(static_cast<uint32_t>(lanes));
    for (int64_t first = 0; first < n; first += most) {
        const int64_t count = n - first < most ? n - first : most;
        const uint32_t per_row = static_cast<uint32_t>(lanes), total = static_cast<uint32_t>(by_rows ? 0 : count * lanes);
        char* const to = out + first * row_bytes;
        const IdT* const from = ids + first;
        if (by_rows) {
            const auto kernel = any ? gather_rows<true, IdT> : gather_rows<false, IdT>;
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(count)), dim3(kBlock), 0, s, w, ldw_bytes, per_row, row_bytes - 16, from, lo, hi, to, row_bytes);
        } else if (vectors) {
            constexpr uint32_t kWidth = kGatherBlock * kGatherVectors;
            const auto kernel = any ? gather_vectors<true, IdT> : gather_vectors<false, IdT>;
            hipLaunchKernelGGL(kernel, dim3((total + kWidth - 1) / kWidth), dim3(kGatherBlock), 0, s, w, ldw_bytes, per_row, div, row_bytes - 16, from, total, lo,
                               hi, to, row_bytes);
        } else {
            const dim3 grid((total + kBlock - 1) / kBlock), block(kBlock);
            if (elem == 1)
                hipLaunchKernelGGL((gather_elements<uint8_t, IdT>), grid, block, 0, s, w, ldw_bytes, per_row, div, from, total, lo, hi, reinterpret_cast<uint8_t*>(to));
            else if (elem == 2)
                hipLaunchKernelGGL((gather_elements<uint16_t, IdT>), grid, block, 0, s, w, ldw_bytes, per_row, div, from, total, lo, hi, reinterpret_cast<uint16_t*>(to));
            else if (elem == 4)
                hipLaunchKernelGGL((gather_elements<uint32_t, IdT>), grid, block, 0, s, w, ldw_bytes, per_row, div, from, total, lo, hi, reinterpret_cast<uint32_t*>(to));
            else
                hipLaunchKernelGGL((gather_elements<uint64_t, IdT>), grid, block, 0, s, w, ldw_bytes, per_row, div, from, total, lo, hi, reinterpret_cast<uint64_t*>(to));
        }
        if (int rc = check_launch("embedding gather")) return rc;
    }
    return 0;
}

__global__ __launch_bounds__(kBlock) void renorm_clear(int32_t* __restrict__ flags, int64_t rows) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < rows) flags[i] = 0;
}

template <typename IdT>
__global__ __launch_bounds__(kBlock) void renorm_mark(const IdT* __restrict__ ids, int64_t n_ids, int64_t lo, int64_t hi,
                                                      int32_t* __restrict__ flags) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= n_ids) return;
    const int64_t id = static_cast<int64_t>(ids[t]);
    if (id >= lo && id < hi) flags[id - lo] = 1;   // every writer stores the same value
}

__device__ inline float wave_max(float v) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, kWave));
    return v;
}

// kind: 1 = sum of magnitudes, 2 = Euclidean, 3 = maximum, 0 = general p.
template <typename T>
__global__ __launch_bounds__(kBlock) void renorm_rows(T* __restrict__ weight, int64_t rows, int64_t dim, int64_t ldw,
                                                      const int32_t* __restrict__ flags, float max_norm, float p, int kind) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + threadIdx.x / kWave;
    if (row >= rows || flags[row] == 0) return;   // the same for all lanes of the wavefront
    T* w = weight + row * ldw;
    float acc = 0.f;
    for (int64_t c = lane; c < dim; c += kWave) {
        const float a = fabsf(load1(w + c));
        if (kind == 1)
            acc += a;
        else if (kind == 2)
            acc += a * a;
        else if (kind == 3)
            acc = fmaxf(acc, a);
        else
            acc += powf(a, p);
    }
    float norm;
    if (kind == 3) {
        norm = wave_max(acc);
    } else {
        const float total = wave_sum(acc);
        norm = kind == 1 ? total : kind == 2 ? sqrtf(total) : powf(total, 1.f / p);
    }
    if (!(norm > max_norm)) return;
    const float scale = max_norm / (norm + 1e-7f);
    for (int64_t c = lane; c < dim; c += kWave) store1(w + c, load1(w + c) * scale);
}

}  // namespace
}  // namespace ddl

extern "C" int ddl_embedding_renorm(void* weight, int dtype, int64_t dim, int64_t ldw, const void* ids, int ids_is_i64,
                                    int64_t n_ids, int64_t lo, int64_t hi, float max_norm, float norm_type, int32_t* flags,
                                    void* stream) {
    using namespace ddl;
    if (dim < 1 || ldw < dim || n_ids < 0 || hi < lo)
        return fail(DDL_E_ARG, "embedding renorm: dim=%lld ldw=%lld n_ids=%lld window=[%lld,%lld)", (long long)dim,
                    (long long)ldw, (long long)n_ids, (long long)lo, (long long)hi);
    if (!(max_norm >= 0.f) || !(norm_type > 0.f))
        return fail(DDL_E_ARG, "embedding renorm: max_norm=%g norm_type=%g", (double)max_norm, (double)norm_type);
    const int64_t rows = hi - lo;
    if (n_ids == 0 || rows == 0) return 0;
    if (!weight || !ids || !flags) return fail(DDL_E_ARG, "embedding renorm: null pointer");
    if (!aligned_to(ids, ids_is_i64 ? 8 : 4) || !aligned_to(flags, 4)) return fail(DDL_E_ALIGN, "embedding renorm: ids or flags misaligned");
    const int64_t row_blocks = (rows + kWavesPerBlock - 1) / kWavesPerBlock, id_blocks = (n_ids + kBlock - 1) / kBlock;
    if (row_blocks > 0x7FFFFFFFll || id_blocks > 0x7FFFFFFFll) return fail(DDL_E_UNSUPP, "embedding renorm: too many rows or ids for one call");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int kind = norm_type == 1.f ? 1 : norm_type == 2.f ? 2 : std::isinf(norm_type) ? 3 : 0;
    int rc = 0;
    const bool known = with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        if (!aligned_to(weight, sizeof(T))) {
            rc = fail(DDL_E_ALIGN, "embedding renorm: table not aligned to its element size");
            return;
        }
        hipLaunchKernelGGL(renorm_clear, dim3(static_cast<uint32_t>((rows + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, flags, rows);
        if (ids_is_i64)
            hipLaunchKernelGGL(renorm_mark<int64_t>, dim3(static_cast<uint32_t>(id_blocks)), dim3(kBlock), 0, s,
                               static_cast<const int64_t*>(ids), n_ids, lo, hi, flags);
        else
            hipLaunchKernelGGL(renorm_mark<int32_t>, dim3(static_cast<uint32_t>(id_blocks)), dim3(kBlock), 0, s,
                               static_cast<const int32_t*>(ids), n_ids, lo, hi, flags);
        hipLaunchKernelGGL(renorm_rows<T>, dim3(static_cast<uint32_t>(row_blocks)), dim3(kBlock), 0, s, static_cast<T*>(weight), rows,
                           dim, ldw, flags, max_norm, norm_type, kind);
        rc = check_launch("renorm_rows");
    });
    if (!known) return fail(DDL_E_UNSUPP, "embedding renorm: dtype %d (f32, bf16 and f16 only)", dtype);
    return rc;
}

extern "C" int ddl_embedding_gather(const void* weight, int64_t dim, int64_t ldw, int elem_size, const void* ids,
                                    int ids_is_i64, int64_t n_ids, int64_t lo, int64_t hi, void* out, void* stream) {
    using namespace ddl;
    if (dim < 1 || ldw < dim || n_ids < 0 || hi < lo)
        return fail(DDL_E_ARG, "embedding gather: dim=%lld ldw=%lld n_ids=%lld window=[%lld,%lld)", (long long)dim,
                    (long long)ldw, (long long)n_ids, (long long)lo, (long long)hi);
    if (elem_size != 1 && elem_size != 2 && elem_size != 4 && elem_size != 8)
        return fail(DDL_E_ARG, "embedding gather: element size %d not in {1,2,4,8}", elem_size);
    if (n_ids == 0) return 0;
    if (!ids || !out || (!weight && hi > lo)) return fail(DDL_E_ARG, "embedding gather: null pointer");
    if (!aligned_to(ids, ids_is_i64 ? 8 : 4)) return fail(DDL_E_ALIGN, "embedding gather: ids misaligned");
    if (!aligned_to(out, elem_size) || !aligned_to(weight, elem_size))
        return fail(DDL_E_ALIGN, "embedding gather: table or output not aligned to the element size");
    const int64_t row_bytes = dim * elem_size, ldw_bytes = ldw * elem_size;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const char* const w = static_cast<const char*>(weight);
    char* const to = static_cast<char*>(out);
    if (ids_is_i64) return launch_gather(w, ldw_bytes, row_bytes, elem_size, static_cast<const int64_t*>(ids), n_ids, lo, hi, to, s);
    return launch_gather(w, ldw_bytes, row_bytes, elem_size, static_cast<const int32_t*>(ids), n_ids, lo, hi, to, s);
}
