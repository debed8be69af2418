// Backward of the DistributedEmbedding shard gather: the adjoint of
// torch.nn.functional.embedding on the local table (reference:
// nn/embedding.py:244-246),
//
//   dweight[r, :] = sum over the tokens t with ids[t] - lo == r of dy[t, :]
//
// for the rows r of the shard window [lo, hi); tokens outside the window and
// tokens equal to padding_idx contribute nothing.  No atomics on the gradient:
// the tokens are first bucketed by table row, then every bucket's dy rows are
// added in fp32, in ascending token order, and every element of dweight is
// written exactly once -- rows nobody looked up get their zeros from the same
// pass, so dweight needs no clearing.
//
//   emb_bwd_clear    counters = 0
//   emb_bwd_count    count[row]++ per token in the window
//   emb_bwd_place    a stretch of the bucket array for every row.  The stretches lie in no particular order, so
//                    no prefix sum over the whole table is needed: a workgroup scans its own 1024 counters and takes its
//                    place with one atomic.  Rows of more than kHotAbove tokens go on the list of hot rows.
//   emb_bwd_fill     bucket[end[row]++] = t
//   emb_bwd_hot      the sums of hot rows: a workgroup per row and 256 bytes of columns (hot_row); not launched
//                    when there are too few tokens for a hot row
//   emb_bwd_reduce   the sums of all other rows: one wavefront (half a wavefront for narrow tables) per row and group
//                    of columns, the bucket ordered in registers
//
// The order in which the fill kernel's atomics hand out bucket slots varies
// from run to run; the reduce kernel orders every bucket so that the fp32 sums
// do not.
//
// What bounds it: the gradient rows read once and the table written once, plus
// the four short kernels in front (2-5 us each, launch and memory latency).
// Token ids as they occur in text make a few rows hot: of 8192 tokens over
// 50304 rows with ids distributed log-uniformly, 483 share one row.  A single
// wavefront walking that bucket one token at a time -- a memory round trip per
// token -- took 1140 us for [50304,512] fp32 where the whole call can take 25.
#include "ddl_common.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

// Workspace of ddl_embedding_backward_static: the counters, bucket cursors, bucket starts and
// token buckets of one call, for callers that cannot hand over (or allocate)
// device memory.  Every GPU the library runs on holds its own 4 MiB copy until
// the process ends; its device address is looked up once per device.
static __device__ __align__(256) int32_t scratch[DDL_EMBEDDING_BACKWARD_STATIC_MAX_ELEMS];

namespace ddl {
namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;

__global__ __launch_bounds__(kBlock) void emb_bwd_clear(int32_t* __restrict__ count, int64_t rows, int32_t* __restrict__ totals) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < rows) count[i] = 0;
    if (i < 2) totals[i] = 0;
}

template <typename IdT>
__device__ inline int64_t token_row(const IdT* __restrict__ ids, int64_t t, int64_t lo, int64_t hi, int64_t padding_idx) {
    const int64_t id = static_cast<int64_t>(ids[t]);
    return (id >= lo && id < hi && id != padding_idx) ? id - lo : -1;
}

// The lanes of a wavefront whose tokens share a row take their places with one
// atomic: `first` receives the lane that issues it, `before` the number of such
// lanes below this one, and the number of such lanes is returned.  Ids as in text
// put hundreds of tokens on one counter, which serves them one after the other
// (8192 such tokens over 50304 rows: count and fill 10 + 11 us without this).
__device__ inline int same_row_lanes(int32_t row, bool on, int lane, int* first, int* before) {
    uint64_t todo = __ballot(on);
    int size = 0;
    *first = lane, *before = 0;
    while (todo) {                                    // the same in all lanes
        const int leader = __ffsll(static_cast<unsigned long long>(todo)) - 1;
        const int32_t r = __builtin_amdgcn_readlane(row, leader);
        const uint64_t same = __ballot(row == r) & todo;
        if ((same >> lane) & 1) {
            *first = leader;
            *before = __popcll(same & ((1ull << lane) - 1));
            size = __popcll(same);
        }
        todo &= ~same;
    }
    return size;
}

template <typename IdT>
__global__ __launch_bounds__(kBlock) void emb_bwd_count(const IdT* __restrict__ ids, int64_t n_ids, int64_t lo, int64_t hi,
                                                        int64_t padding_idx, int32_t* __restrict__ count) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const int32_t r = t < n_ids ? static_cast<int32_t>(token_row(ids, t, lo, hi, padding_idx)) : -1;
    const int lane = threadIdx.x & (kWave - 1);
    int first, before;
    const int size = same_row_lanes(r, r >= 0, lane, &first, &before);
    if (r >= 0 && before == 0) atomicAdd(&count[r], size);
}

// Stretches of the bucket array.  end[row] is where the row's stretch begins;
// the fill kernel advances it to where it ends.  totals[0]: slots handed out so
// far, totals[1]: entries of the hot list.  The last row of the table never goes
// on the list (it is looked at in any case), so the list has at most rows - 1 entries.
constexpr int kPlaceRows = 4;                     // consecutive rows of a thread
__global__ __launch_bounds__(kBlock) void emb_bwd_place(const int32_t* __restrict__ count, int64_t rows, int32_t hot_above,
                                                        int32_t* __restrict__ end, int32_t* __restrict__ hot, int32_t* __restrict__ totals) {
    __shared__ int32_t wave_total[kWavesPerBlock];
    __shared__ int32_t base;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * kPlaceRows;
    int32_t n[kPlaceRows], total = 0;
#pragma unroll
    for (int k = 0; k < kPlaceRows; ++k) {
        n[k] = r0 + k < rows ? count[r0 + k] : 0;
        total += n[k];
    }
    int32_t incl = total;                                      // inclusive scan over the wavefront
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t up = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += up;
    }
    if (lane == kWave - 1) wave_total[wave] = incl;
    __syncthreads();
    int32_t before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < kWavesPerBlock; ++k) {
        before += k < wave ? wave_total[k] : 0;
        all += wave_total[k];
    }
    if (threadIdx.x == 0) base = all ? atomicAdd(&totals[0], all) : 0;
    __syncthreads();
    int32_t run = base + before + incl - total;
#pragma unroll
    for (int k = 0; k < kPlaceRows; ++k) {
        if (r0 + k >= rows) break;
        end[r0 + k] = run;
        run += n[k];
        if (n[k] > hot_above && r0 + k < rows - 1) hot[atomicAdd(&totals[1], 1)] = static_cast<int32_t>(r0 + k);
    }
}

template <typename IdT>
__global__ __launch_bounds__(kBlock) void emb_bwd_fill(const IdT* __restrict__ ids, int64_t n_ids, int64_t lo, int64_t hi,
                                                       int64_t padding_idx, int32_t* __restrict__ end, int32_t* __restrict__ bucket) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const int32_t r = t < n_ids ? static_cast<int32_t>(token_row(ids, t, lo, hi, padding_idx)) : -1;
    const int lane = threadIdx.x & (kWave - 1);
    int first, before;
    const int size = same_row_lanes(r, r >= 0, lane, &first, &before);
    int32_t slot = 0;
    if (r >= 0 && before == 0) slot = atomicAdd(&end[r], size);
    slot = __shfl(slot, first, kWave) + before;
    if (r >= 0) bucket[slot] = static_cast<int32_t>(t);
}

// Elements: bf16 or fp16 bits or float; all are summed in fp32 and rounded once on the way out.
struct Bf16 {
    typedef uint16_t word;
    static __device__ float widen(uint16_t u) { return __uint_as_float(static_cast<uint32_t>(u) << 16); }
    static __device__ uint16_t round(float f) {
        const __bf16 b = static_cast<__bf16>(f);
        uint16_t u;
        __builtin_memcpy(&u, &b, 2);
        return u;
    }
};
struct F16 {
    typedef uint16_t word;
    static __device__ float widen(uint16_t u) {
        _Float16 h;
        __builtin_memcpy(&h, &u, 2);
        return static_cast<float>(h);
    }
    static __device__ uint16_t round(float f) {
        const _Float16 h = static_cast<_Float16>(f);
        uint16_t u;
        __builtin_memcpy(&u, &h, 2);
        return u;
    }
};
struct F32 {
    typedef float word;
    static __device__ float widen(float f) { return f; }
    static __device__ float round(float f) { return f; }
};

// V consecutive elements in one access, aligned to an element only (gfx950 serves
// 16-byte accesses at any alignment, and a copy of rows of odd length runs at
// nine tenths of the aligned rate).
template <typename W, int V>
struct Pack {
    W e[V];
};
template <typename W, int V>
__device__ inline Pack<W, V> load_pack(const W* p) {
    typedef W raw __attribute__((ext_vector_type(V)));
    typedef raw loose __attribute__((aligned(sizeof(W))));
    const raw r = *reinterpret_cast<const loose*>(p);
    Pack<W, V> out;
    __builtin_memcpy(&out, &r, sizeof(out));
    return out;
}
template <typename W, int V>
__device__ inline void store_pack(W* p, const Pack<W, V>& v) {   // streaming: the gradient is not read again here
    typedef W raw __attribute__((ext_vector_type(V)));
    typedef raw loose __attribute__((aligned(sizeof(W))));
    raw r;
    __builtin_memcpy(&r, &v, sizeof(r));
    __builtin_nontemporal_store(r, reinterpret_cast<loose*>(p));
}

struct ReduceArgs {
    const void* dy;
    void* dw;
    int64_t dim, ld_dy, ld_dw, rows;
    const int32_t* count;
    const int32_t* end;
    const int32_t* bucket;
    const int32_t* hot;
    const int32_t* totals;
    int64_t n_ids;
    int32_t nv;             // vectors of V elements per row; the last one is moved back to end with the row
    int32_t passes;         // groups of columns per row of the ordinary path
    int32_t rows_per_block;
    int32_t hot_above;      // rows of more tokens are hot
    int32_t hot_chunks;     // 256-byte pieces of a row
    int32_t scale_by_freq;
};

// ---- hot rows ----
// A workgroup owns 256 bytes of columns of one row.  What takes time is the
// memory round trip, not the additions, so all threads fetch the pieces of the
// next two batches of 64 tokens -- 16 lanes a token, 16 bytes a lane -- while one
// wavefront adds a batch in token order out of LDS, a column (or two 16-bit ones)
// per lane: the sums stay strictly sequential per column with 128 tokens in
// flight.  (A wavefront that walks its columns alone keeps 32 in flight in the
// same registers: 55 us instead of 20 for 483 tokens of 2 KiB.)
// The order of the tokens: up to 512 by counting the smaller ones, more through
// a bit per token number in LDS (16 KiB for a window of 131072 of them) that is
// read back in ascending order, kListTokens at a time.  The bits have LDS of their
// own: in the stage's they had to be set again, by a walk over the whole bucket,
// for every kListTokens (2^20 tokens of one row, 256 bytes each: 1267 ms, now 59).
constexpr int kHotAbove = 32;                        // rows of more tokens are hot: what half a wavefront's lanes order, and as long as
                                                     // the ordinary walk stays below the time of everything else (with 64: 24 us, with 32: 17)
constexpr int kHotBytes = 256;
constexpr int kHotBatch = 64;                        // tokens per batch
constexpr int kListTokens = 1024;
constexpr int kRankTokens = 2 * kBlock;
constexpr int kBitWords = 4096;
constexpr int kBitsPerWindow = kBitWords * 32;
constexpr int kWordsPerThread = kBitWords / kBlock;

struct HotShared {
    uint32_t pieces[kHotBytes * kHotBatch / 4];      // of a batch
    uint32_t bits[kBitWords];                        // a bit per token number, or the bucket being ordered
    int32_t list[kListTokens];                       // tokens in ascending order
    int32_t wave_total[kWavesPerBlock];
};

// Adds the first m tokens of the list to the columns from col0 on; called by all threads.
template <typename E>
__device__ inline void hot_accumulate(HotShared& sh, const ReduceArgs& a, int64_t col0, int m, float (&acc)[2]) {
    typedef typename E::word W;
    constexpr int V = 16 / sizeof(W);
    constexpr int kLanesPerToken = 16, kTokensPerLoad = kBlock / kLanesPerToken, kLoads = kHotBatch / kTokensPerLoad;
    const int t = threadIdx.x, part = t % kLanesPerToken, tok0 = t / kLanesPerToken;
    const int64_t col = col0 + part * V, left = a.dim - col;
    const W* const dy = static_cast<const W*>(a.dy) + col;
    uint4 piece[2][kLoads];
    auto fetch = [&](uint4 (&to)[kLoads], int base) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int i = base + u * kTokensPerLoad + tok0;
            to[u] = make_uint4(0, 0, 0, 0);
            if (i >= m || left <= 0) continue;
            const W* src = dy + static_cast<int64_t>(sh.list[i]) * a.ld_dy;
            Pack<W, V> v;
            if (left >= V) {
                v = load_pack<W, V>(src);
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) v.e[e] = e < left ? src[e] : W(0);
            }
            __builtin_memcpy(&to[u], &v, 16);
        }
    };
    auto batch = [&](uint4 (&from)[kLoads], int base) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
            *reinterpret_cast<uint4*>(&sh.pieces[(u * kTokensPerLoad + tok0) * (kHotBytes / 4) + part * 4]) = from[u];
        __syncthreads();
        if (base + 2 * kHotBatch < m) fetch(from, base + 2 * kHotBatch);
        if (t < kWave) {
            const int here = m - base < kHotBatch ? m - base : kHotBatch;
            auto add = [&](uint32_t w) {
                if constexpr (sizeof(W) == 4) {
                    acc[0] += __uint_as_float(w);
                } else {
                    acc[0] += E::widen(static_cast<uint16_t>(w));
                    acc[1] += E::widen(static_cast<uint16_t>(w >> 16));
                }
            };
            int k = 0;
            for (; k + 16 <= here; k += 16) {
                uint32_t w[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) w[u] = sh.pieces[(k + u) * (kHotBytes / 4) + t];
#pragma unroll
                for (int u = 0; u < 16; ++u) add(w[u]);
            }
            for (; k < here; ++k) add(sh.pieces[k * (kHotBytes / 4) + t]);
        }
        __syncthreads();
    };
    fetch(piece[0], 0);
    if (kHotBatch < m) fetch(piece[1], kHotBatch);
    for (int base = 0; base < m; base += 2 * kHotBatch) {
        batch(piece[0], base);
        if (base + kHotBatch < m) batch(piece[1], base + kHotBatch);
    }
}

// Called by every thread of the workgroup with the same arguments.
template <typename E>
__device__ inline void hot_row(HotShared& sh, const ReduceArgs& a, int64_t row, int chunk) {
    typedef typename E::word W;
    const int32_t n = a.count[row];
    const int32_t* const bucket = a.bucket + (a.end[row] - n);
    const int t = threadIdx.x;
    const int64_t col0 = static_cast<int64_t>(chunk) * (kHotBytes / sizeof(W));
    float acc[2] = {0.f, 0.f};
    if (n <= kRankTokens) {
        int32_t* const raw = reinterpret_cast<int32_t*>(sh.bits);
        // two tokens per thread; INT_MAX behind the bucket's end is smaller than nothing
        const int32_t t0 = t < n ? bucket[t] : 0x7FFFFFFF, t1 = t + kBlock < n ? bucket[t + kBlock] : 0x7FFFFFFF;
        raw[t] = t0, raw[t + kBlock] = t1;
        __syncthreads();
        int rank0 = 0, rank1 = 0;
#pragma unroll 4
        for (int k = 0; k < n; k += 4) {
            const int4 q = *reinterpret_cast<const int4*>(&raw[k]);
            rank0 += (q.x < t0) + (q.y < t0) + (q.z < t0) + (q.w < t0);
            rank1 += (q.x < t1) + (q.y < t1) + (q.z < t1) + (q.w < t1);
        }
        if (t < n) sh.list[rank0] = t0;
        if (t + kBlock < n) sh.list[rank1] = t1;
        __syncthreads();
        hot_accumulate<E>(sh, a, col0, n, acc);
    } else {
        const int lane = t & (kWave - 1), wave = t / kWave;
        for (int64_t w0 = 0; w0 < a.n_ids; w0 += kBitsPerWindow) {
            for (int i = t; i < kBitWords; i += kBlock) sh.bits[i] = 0;
            __syncthreads();
#pragma unroll 4
            for (int32_t i = t; i < n; i += kBlock) {
                const int64_t at = bucket[i] - w0;
                if (at >= 0 && at < kBitsPerWindow) atomicOr(&sh.bits[at >> 5], 1u << (at & 31));
            }
            __syncthreads();
            int32_t mine = 0;
            for (int k = 0; k < kWordsPerThread; ++k) mine += __popc(sh.bits[t * kWordsPerThread + k]);
            int32_t incl = mine;
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const int32_t up = __shfl_up(incl, off, kWave);
                if (lane >= off) incl += up;
            }
            if (lane == kWave - 1) sh.wave_total[wave] = incl;
            __syncthreads();
            int32_t rank0 = incl - mine, in_window = 0;
#pragma unroll
            for (int k = 0; k < kWavesPerBlock; ++k) {
                rank0 += k < wave ? sh.wave_total[k] : 0;
                in_window += sh.wave_total[k];
            }
            for (int32_t first = 0; first < in_window; first += kListTokens) {   // the same in all threads
                if (rank0 < first + kListTokens && rank0 + mine > first) {
                    int32_t rank = rank0;
                    for (int k = 0; k < kWordsPerThread; ++k) {
                        uint32_t bits = sh.bits[t * kWordsPerThread + k];
                        while (bits) {
                            const int b = __ffs(bits) - 1;
                            bits &= bits - 1;
                            if (rank >= first && rank < first + kListTokens)
                                sh.list[rank - first] = static_cast<int32_t>(w0) + (t * kWordsPerThread + k) * 32 + b;
                            ++rank;
                        }
                    }
                }
                __syncthreads();
                const int32_t here = in_window - first;
                hot_accumulate<E>(sh, a, col0, here < kListTokens ? here : kListTokens, acc);
            }
        }
    }
    if (t < kWave) {
        const float scale = (a.scale_by_freq && n > 1) ? 1.0f / static_cast<float>(n) : 1.0f;
        W* const dst = static_cast<W*>(a.dw) + row * a.ld_dw + col0;
        if constexpr (sizeof(W) == 4) {
            if (col0 + t < a.dim) dst[t] = acc[0] * scale;
        } else {
            if (col0 + 2 * t < a.dim) dst[2 * t] = E::round(acc[0] * scale);
            if (col0 + 2 * t + 1 < a.dim) dst[2 * t + 1] = E::round(acc[1] * scale);
        }
    }
    __syncthreads();                                 // the list is rewritten by the workgroup's next row
}

// A launch of its own: with the hot rows' registers and LDS the ordinary rows,
// which live on many wavefronts, took 64 us instead of 50 for [16032,4096] bf16.
template <typename E>
__global__ __launch_bounds__(kBlock) void emb_bwd_hot(const ReduceArgs a) {
    __shared__ HotShared sh;
    // the list, and the last row of the table if it is hot
    const int32_t listed = a.totals[1];
    const int32_t items = (listed + (a.count[a.rows - 1] > a.hot_above ? 1 : 0)) * a.hot_chunks;
    for (int32_t item = static_cast<int32_t>(blockIdx.x); item < items; item += static_cast<int32_t>(gridDim.x)) {
        const int32_t which = item / a.hot_chunks;
        hot_row<E>(sh, a, which < listed ? a.hot[which] : a.rows - 1, item - which * a.hot_chunks);
    }
}

// ---- ordinary rows ----
// V: elements per vector (16 bytes, or 1 for rows shorter than that).  LPR lanes
// share a row (32: two rows per wavefront, for rows of at most 32 vectors), CPW
// vectors per lane and pass.  Buckets (of at most kHotAbove tokens) are ordered in
// registers: lane i holds one token, counts the smaller ones (its rank) and sends
// it to the lane of that number (lanes without a token send theirs, larger than
// any, to the lane behind the last).
template <typename E, int V, int LPR, int CPW>
__global__ __launch_bounds__(kBlock, 8) void emb_bwd_reduce(const ReduceArgs a) {
    typedef typename E::word W;
    constexpr int kGroups = kWave / LPR;
    const int lane = threadIdx.x & (kWave - 1), g = lane / LPR, gl = lane % LPR;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * a.rows_per_block;
    const int items = a.rows_per_block / kGroups * a.passes;
    const W* const dy = static_cast<const W*>(a.dy);
    for (int item = threadIdx.x / kWave; item < items; item += kWavesPerBlock) {
        const int q = item / a.passes, pass = item - q * a.passes;
        const int64_t row = row0 + q * kGroups + g;
        const bool real = row < a.rows;
        int32_t n = real ? a.count[row] : 0;
        const bool mine_to_write = real && n <= a.hot_above;
        if (!mine_to_write) n = 0;
        int32_t m = __builtin_amdgcn_readlane(n, 0);
        if (kGroups == 2) {
            const int32_t m1 = __builtin_amdgcn_readlane(n, kWave - 1);
            m = m > m1 ? m : m1;
        }
        float acc[CPW][V];
#pragma unroll
        for (int j = 0; j < CPW; ++j)
#pragma unroll
            for (int e = 0; e < V; ++e) acc[j][e] = 0.f;
        int64_t col[CPW];
        bool on[CPW];
#pragma unroll
        for (int j = 0; j < CPW; ++j) {
            const int64_t v = static_cast<int64_t>(pass) * (LPR * CPW) + j * LPR + gl;
            on[j] = v < a.nv;
            col[j] = v * V;
            if (col[j] > a.dim - V) col[j] = a.dim - V;          // the last vector ends with the row (or a lane has none)
        }
        if (m > 0) {                                             // the same in all lanes
            int32_t tok = gl < n ? a.bucket[a.end[row] - n + gl] : 0x7FFFFFFF;
            if (m > 1) {
                int rank = 0;
                for (int k = 0; k < m; ++k) rank += __shfl(tok, g * LPR + k, kWave) < tok ? 1 : 0;
                tok = __builtin_amdgcn_ds_permute((g * LPR + rank) << 2, tok);
            }
            auto add_tokens = [&](int k0, auto count) {
                constexpr int U = decltype(count)::value;
                Pack<W, V> v[U][CPW];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int32_t at = __shfl(tok, g * LPR + k0 + u, kWave);
                    const W* src = dy + static_cast<int64_t>(kGroups == 1 || k0 + u < n ? at : 0) * a.ld_dy;   // token 0 exists
#pragma unroll
                    for (int j = 0; j < CPW; ++j) v[u][j] = load_pack<W, V>(src + col[j]);
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int j = 0; j < CPW; ++j)
#pragma unroll
                        for (int e = 0; e < V; ++e) acc[j][e] += (kGroups == 1 || k0 + u < n) ? E::widen(v[u][j].e[e]) : 0.f;
            };
            int k = 0;
            constexpr int kMost = (CPW == 1 ? 4 : 2) * (sizeof(W) == 4 ? 2 : 1);   // what 64 registers hold
            for (; k + kMost <= m; k += kMost) add_tokens(k, std::integral_constant<int, kMost>{});
            if (kMost > 4 && k + 4 <= m) {
                add_tokens(k, std::integral_constant<int, 4>{});
                k += 4;
            }
            if (kMost > 2 && k + 2 <= m) {
                add_tokens(k, std::integral_constant<int, 2>{});
                k += 2;
            }
            if (k < m) add_tokens(k, std::integral_constant<int, 1>{});
        }
        if (!mine_to_write) continue;
        W* const dst = static_cast<W*>(a.dw) + row * a.ld_dw;
        const float scale = (a.scale_by_freq && n > 1) ? 1.0f / static_cast<float>(n) : 1.0f;
#pragma unroll
        for (int j = 0; j < CPW; ++j) {
            if (!on[j]) continue;
            Pack<W, V> o;
#pragma unroll
            for (int e = 0; e < V; ++e) o.e[e] = E::round(acc[j][e] * scale);
            store_pack<W, V>(dst + col[j], o);
        }
    }
}

template <typename E, int V>
void launch_reduce(ReduceArgs a, hipStream_t s) {
    a.nv = static_cast<int32_t>((a.dim + V - 1) / V);
    auto go = [&](auto kernel, int lpr, int cpw) {
        a.passes = (a.nv + lpr * cpw - 1) / (lpr * cpw);
        // One row per workgroup when a row has work for three or four wavefronts, else as many rows as fill them.
        a.rows_per_block = a.passes >= 3 ? 1 : (kWave / lpr) * (kWavesPerBlock / a.passes);
        const int64_t blocks = (a.rows + a.rows_per_block - 1) / a.rows_per_block;
        hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kBlock), 0, s, a);
    };
    if (a.nv <= 32)
        go(emb_bwd_reduce<E, V, 32, 1>, 32, 1);
    else if (a.nv <= 64)
        go(emb_bwd_reduce<E, V, 64, 1>, 64, 1);
    else
        go(emb_bwd_reduce<E, V, 64, 2>, 64, 2);
}

template <typename E>
void launch_reduce_any(const ReduceArgs& a, uint32_t hot_blocks, hipStream_t s) {
    constexpr int V = 16 / sizeof(typename E::word);
    if (hot_blocks > 0) hipLaunchKernelGGL(emb_bwd_hot<E>, dim3(hot_blocks), dim3(kBlock), 0, s, a);
    if (a.dim >= V)
        launch_reduce<E, V>(a, s);
    else
        launch_reduce<E, 1>(a, s);
}

template <typename IdT>
int run(const void* dy, int dtype, int64_t dim, int64_t ld_dy, const IdT* ids, int64_t n_ids, int64_t lo, int64_t hi,
        int64_t padding_idx, int scale_by_freq, void* dw, int64_t ld_dw, int32_t* ws, hipStream_t s) {
    const int64_t rows = hi - lo;
    const int es = dtype == DDL_DT_F32 ? 4 : 2;
    ReduceArgs a{};
    a.dy = dy, a.dw = dw, a.dim = dim, a.ld_dy = ld_dy, a.ld_dw = ld_dw, a.rows = rows, a.n_ids = n_ids;
    a.scale_by_freq = scale_by_freq;
    a.hot_above = kHotAbove;
    // 3 rows + 1 + n_ids integers: the hot list has at most rows - 1 entries
    int32_t* const count = ws;                              // [rows]      tokens of each row
    int32_t* const end = ws + rows;                         // [rows]      next free slot of each row's stretch
    int32_t* const totals = end + rows;                     // [2]
    int32_t* const bucket = totals + 2;                     // [n_ids]
    int32_t* const hot = bucket + n_ids;                    // [rows - 1]
    a.count = count, a.end = end, a.bucket = bucket, a.hot = hot, a.totals = totals;
    const int64_t most_hot = std::min(rows, n_ids / (a.hot_above + 1));
    a.hot_chunks = static_cast<int32_t>((dim * es + kHotBytes - 1) / kHotBytes);
    const uint32_t hot_blocks = static_cast<uint32_t>(std::min<int64_t>(most_hot * a.hot_chunks, 1024));
    auto grid = [](int64_t n) { return dim3(static_cast<uint32_t>((n + kBlock - 1) / kBlock)); };
    hipLaunchKernelGGL(emb_bwd_clear, grid(std::max<int64_t>(rows, 2)), dim3(kBlock), 0, s, count, rows, totals);
    if (n_ids > 0) {
        hipLaunchKernelGGL((emb_bwd_count<IdT>), grid(n_ids), dim3(kBlock), 0, s, ids, n_ids, lo, hi, padding_idx, count);
        hipLaunchKernelGGL(emb_bwd_place, grid((rows + kPlaceRows - 1) / kPlaceRows), dim3(kBlock), 0, s, count, rows, a.hot_above, end, hot, totals);
        hipLaunchKernelGGL((emb_bwd_fill<IdT>), grid(n_ids), dim3(kBlock), 0, s, ids, n_ids, lo, hi, padding_idx, end, bucket);
    }
    if (dtype == DDL_DT_F16)
        launch_reduce_any<F16>(a, hot_blocks, s);
    else if (dtype == DDL_DT_BF16)
        launch_reduce_any<Bf16>(a, hot_blocks, s);
    else
        launch_reduce_any<F32>(a, hot_blocks, s);
    return check_launch("embedding backward");
}

constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
int32_t* scratch_address[kMaxDevices] = {};   // device address of `scratch` on each GPU, filled on first use

// The device address of `scratch` on the current GPU.  In host code the name
// `scratch` is only a handle for the runtime, never a pointer a kernel may use.
int scratch_on_current_device(int32_t** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(static_cast<int>(e), "embedding backward (static): hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(DDL_E_UNSUPP, "embedding backward (static): device index %d (at most %d devices)", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_address[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(e != hipSuccess ? static_cast<int>(e) : DDL_E_ARG, "embedding backward (static): hipGetSymbolAddress: %s", hipGetErrorString(e));
        scratch_address[dev] = static_cast<int32_t*>(p);
    }
    *out = scratch_address[dev];
    return 0;
}

}  // namespace
}  // namespace ddl

extern "C" int ddl_embedding_backward_static(const void* dy, int dtype, int64_t dim, int64_t ld_dy, const void* ids, int ids_is_i64,
                                             int64_t n_ids, int64_t lo, int64_t hi, int64_t padding_idx, int scale_grad_by_freq,
                                             void* dweight, int64_t ld_dw, void* stream) {
    using namespace ddl;
    if (n_ids < 0 || hi < lo) return fail(DDL_E_ARG, "embedding backward (static): n_ids=%lld window=[%lld,%lld)", (long long)n_ids, (long long)lo, (long long)hi);
    const int64_t rows = hi - lo;
    // compared without forming 2 rows + 1 + n_ids, which could overflow
    if (rows > DDL_EMBEDDING_BACKWARD_STATIC_MAX_ELEMS || n_ids > DDL_EMBEDDING_BACKWARD_STATIC_MAX_ELEMS ||
        3 * rows + 1 + n_ids > DDL_EMBEDDING_BACKWARD_STATIC_MAX_ELEMS)
        return fail(DDL_E_UNSUPP,
                    "embedding backward (static): 3 * %lld rows + 1 + %lld tokens exceeds the built-in workspace of %lld int32; "
                    "use ddl_embedding_backward with a workspace of your own", (long long)rows, (long long)n_ids,
                    (long long)DDL_EMBEDDING_BACKWARD_STATIC_MAX_ELEMS);
    int32_t* ws = nullptr;
    const int rc = scratch_on_current_device(&ws);
    if (rc) return rc;
    return ddl_embedding_backward(dy, dtype, dim, ld_dy, ids, ids_is_i64, n_ids, lo, hi, padding_idx, scale_grad_by_freq, dweight,
                                  ld_dw, ws, DDL_EMBEDDING_BACKWARD_STATIC_MAX_ELEMS, stream);
}

extern "C" int ddl_embedding_backward(const void* dy, int dtype, int64_t dim, int64_t ld_dy, const void* ids, int ids_is_i64,
                                      int64_t n_ids, int64_t lo, int64_t hi, int64_t padding_idx, int scale_grad_by_freq,
                                      void* dweight, int64_t ld_dw, int32_t* workspace, int64_t workspace_elems, void* stream) {
    using namespace ddl;
    if (dim < 0 || ld_dy < dim || ld_dw < dim || n_ids < 0 || hi < lo)
        return fail(DDL_E_ARG, "embedding backward: dim=%lld ld_dy=%lld ld_dw=%lld n_ids=%lld window=[%lld,%lld)", (long long)dim,
                    (long long)ld_dy, (long long)ld_dw, (long long)n_ids, (long long)lo, (long long)hi);
    if (dtype != DDL_DT_BF16 && dtype != DDL_DT_F16 && dtype != DDL_DT_F32)
        return fail(DDL_E_UNSUPP, "embedding backward: dtype %d (bf16, f16 and f32 only)", dtype);
    const int64_t rows = hi - lo;
    if (rows == 0 || dim == 0) return 0;
    if (n_ids > 0x7FFFFFFFll || rows > 0x3FFFFFFFll) return fail(DDL_E_UNSUPP, "embedding backward: more than 2^31 tokens or 2^30 rows");
    if (!dweight || !workspace || (n_ids > 0 && (!dy || !ids))) return fail(DDL_E_ARG, "embedding backward: null pointer");
    const int es = dtype == DDL_DT_F32 ? 4 : 2;
    if (!aligned_to(dy, es) || !aligned_to(dweight, es) || !aligned_to(workspace, 4) || !aligned_to(ids, ids_is_i64 ? 8 : 4))
        return fail(DDL_E_ALIGN, "embedding backward: pointer misaligned");
    const int64_t need = 3 * rows + 1 + n_ids;
    if (workspace_elems < need)
        return fail(DDL_E_ARG, "embedding backward: workspace of %lld int32 is smaller than the %lld needed (3 rows + 1 + tokens)",
                    (long long)workspace_elems, (long long)need);
    const int64_t chunks = (dim + 63) / 64;
    if (rows >= 0x7FFFFFFFll || chunks > 0xFFFFFF) return fail(DDL_E_UNSUPP, "embedding backward: too many workgroups or columns");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (ids_is_i64)
        return run(dy, dtype, dim, ld_dy, static_cast<const int64_t*>(ids), n_ids, lo, hi, padding_idx, scale_grad_by_freq != 0, dweight,
                   ld_dw, workspace, s);
    return run(dy, dtype, dim, ld_dy, static_cast<const int32_t*>(ids), n_ids, lo, hi, padding_idx, scale_grad_by_freq != 0, dweight, ld_dw,
               workspace, s);
}
