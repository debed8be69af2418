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
//   emb_bwd_split    tokens of a chunk of ids sorted by segment; segment s owns the rows s, s + G, s + 2 G, ... of the
//                    table (frequent ids are neighbours in a vocabulary sorted by frequency: so they spread)
//   emb_bwd_buckets  a workgroup per segment: counts and places its tokens with counters in LDS.  Nothing has to be cleared,
//                    and a row that many tokens share costs LDS atomics of one workgroup.  Few tokens are read by every
//                    workgroup, without emb_bwd_split in front
//   with less workspace than these take, or a table of more than 2^23 rows, four launches instead:
//   emb_bwd_clear    counters = 0
//   emb_bwd_count    count[row]++ per token in the window
//   emb_bwd_place    a stretch of the bucket array for every row.  The stretches lie in no particular order, so
//                    no prefix sum over the whole table is needed: a workgroup scans its own 1024 counters and takes its
//                    place with one atomic.  Rows of more than kHotAbove tokens go on the list of hot rows.
//   emb_bwd_fill     bucket[end[row]++] = t
//   then
//   emb_bwd_hot      the sums of hot rows: a workgroup per row and 64 bytes of columns (hot_row); not launched
//                    when there are too few tokens for a hot row
//   emb_bwd_reduce   the sums of all other rows: one wavefront (half a wavefront for narrow tables) per row and group
//                    of columns, the bucket ordered in registers
//   emb_bwd_sums     both, after the bucketing by segments of up to 131072 tokens
//
// The order in which atomics hand out bucket slots varies from run to run; the
// kernels that add order every bucket so that the fp32 sums do not.
//
// What bounds it: the gradient rows read once and the table written once, plus
// the short kernels in front (2-5 us each, launch and memory latency).
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

// What is known of a row: its number of tokens, and the end of its stretch of the bucket array.
struct Row {
    int32_t count, end;
};

__global__ __launch_bounds__(kBlock) void emb_bwd_clear(Row* __restrict__ meta, int64_t rows, int32_t* __restrict__ totals) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < rows) meta[i].count = 0;
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
                                                        int64_t padding_idx, Row* __restrict__ meta) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const int32_t r = t < n_ids ? static_cast<int32_t>(token_row(ids, t, lo, hi, padding_idx)) : -1;
    const int lane = threadIdx.x & (kWave - 1);
    int first, before;
    const int size = same_row_lanes(r, r >= 0, lane, &first, &before);
    if (r >= 0 && before == 0) atomicAdd(&meta[r].count, size);
}

// Stretches of the bucket array.  A row's `end` is set to where its stretch begins;
// the fill kernel advances it to where it ends.  totals[0]: slots handed out so
// far, totals[1]: entries of the hot list.  The last row of the table never goes
// on the list (it is looked at in any case), so the list has at most rows - 1 entries.
constexpr int kPlaceRows = 4;                     // consecutive rows of a thread
__global__ __launch_bounds__(kBlock) void emb_bwd_place(Row* __restrict__ meta, int64_t rows, int32_t hot_above, int32_t* __restrict__ hot,
                                                        int32_t* __restrict__ totals) {
    __shared__ int32_t wave_total[kWavesPerBlock];
    __shared__ int32_t base;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * kPlaceRows;
    int32_t n[kPlaceRows], total = 0;
#pragma unroll
    for (int k = 0; k < kPlaceRows; ++k) {
        n[k] = r0 + k < rows ? meta[r0 + k].count : 0;
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
        meta[r0 + k].end = run;
        run += n[k];
        if (n[k] > hot_above && r0 + k < rows - 1) hot[atomicAdd(&totals[1], 1)] = static_cast<int32_t>(r0 + k);
    }
}

template <typename IdT>
__global__ __launch_bounds__(kBlock) void emb_bwd_fill(const IdT* __restrict__ ids, int64_t n_ids, int64_t lo, int64_t hi,
                                                       int64_t padding_idx, Row* __restrict__ meta, int32_t* __restrict__ bucket) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const int32_t r = t < n_ids ? static_cast<int32_t>(token_row(ids, t, lo, hi, padding_idx)) : -1;
    const int lane = threadIdx.x & (kWave - 1);
    int first, before;
    const int size = same_row_lanes(r, r >= 0, lane, &first, &before);
    int32_t slot = 0;
    if (r >= 0 && before == 0) slot = atomicAdd(&meta[r].end, size);
    slot = __shfl(slot, first, kWave) + before;
    if (r >= 0) bucket[slot] = static_cast<int32_t>(t);
}

// ---- bucketing in two launches ----
// Bound by latency: launches, LDS atomics, a few dependent trips to L2.  Measured, four launches -> two: 131072 uniform
// tokens over 128256 ids, 16032 of them rows, 20 -> 10.5 us; as in text (11000 tokens on one row) 92 -> 28 us; 8192 tokens as
// in text over 50304 rows 19 -> 16 us with the buckets left in order, which takes the hot rows' kernel 6 us less; 16 tokens
// 7.6 -> 7.3 us.  Up to kOneTokens tokens one launch, whose workgroups each look at all of them, does (24 us for 131072 tokens, 79 as
// in text).  The whole gradient, two launches -> one: 8192 tokens as in text, [50304, 512] fp32 41.7 -> 39.8 us, 2048 33.3 -> 29.8;
// 4000, [2000, 64] 26.3 -> 22.7; 856, [2538, 1210] bf16 14.7 -> 11.7; 16, [125, 64] 9.7 -> 7.3.
constexpr int kSplitBlock = 256;
constexpr int kBucketBlock = 1024;
constexpr int kChunks = 1024;                     // chunks of tokens, at most
constexpr int kSegmentRows = 4096;                // rows of a segment, at most
constexpr int kSegments = 2048;                   // segments, at most; a power of two from 256 on
constexpr int kHeldTokens = 4096;                 // tokens of a segment that are placed in LDS first
constexpr int kLongRows = 256;
constexpr int32_t kOrdered = 0x40000000;          // in an entry of the hot list: the row's bucket is in ascending order
constexpr int32_t kLong = 0x20000000;             // of the slots of emb_bwd_buckets<.., true>: more than kRankTokens tokens
constexpr int kOneTokens = 8192;                  // bucketed in one launch: up to so many tokens,
constexpr int kOneRows = 1024;                    // 256 segments of up to so many rows
constexpr int kHotSlots = 512;                    // slots of hot rows, at most
constexpr int kRankTokens = 2 * kBlock;           // up to so many tokens of a row are ordered by counting the smaller ones
constexpr int kBitWords = 4096;                   // more of them by a bit per token number
constexpr int kBitsPerWindow = kBitWords * 32;

struct SplitArgs {
    int64_t n_ids, lo, padding_idx, chunk_tokens;
    int32_t rows, segments, shift;                // segments = 1 << shift
    int32_t segment_rows, chunks, hot_above;
    int32_t* offsets;                             // [chunks][segments + 1]: first token of the segment in the chunk
    int32_t* token;                               // [n_ids] tokens of a chunk by segment
    int32_t* row;                                 // [n_ids] their rows inside the segment
    Row* meta;                                    // [segments][segment_rows]
    int32_t* bucket;
    int32_t* hot;
    int32_t* totals;                              // entries at the end of the hot list, entries at its front
    int32_t hot_most;                             // entries the hot list has room for
};

// Slots of hot rows that the segments up to one whose tokens end at `tokens` have: one for every kHotAbove + 1 tokens and one
// more for each segment.
constexpr int kHotAbove = 32;                        // rows of more tokens are hot: what half a wavefront's lanes order, and as long as
                                                     // the ordinary walk stays below the time of everything else (with 64: 24 us, with 32: 17)
__host__ __device__ inline int32_t hot_slots(int32_t tokens, int32_t segments) { return tokens / (kHotAbove + 1) + segments; }

template <typename IdT>
__global__ __launch_bounds__(kSplitBlock) void emb_bwd_split(const IdT* __restrict__ ids, const SplitArgs a) {
    __shared__ int32_t cursor[kSegments];
    __shared__ int32_t wave_total[kSplitBlock / kWave];
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
    const int64_t t0 = blockIdx.x * a.chunk_tokens, t1 = t0 + a.chunk_tokens < a.n_ids ? t0 + a.chunk_tokens : a.n_ids;
    for (int s = t; s < a.segments; s += kSplitBlock) cursor[s] = 0;
    if (blockIdx.x == 0 && t < 2) a.totals[t] = 0;
    __syncthreads();
    for (int64_t i = t0 + t; i < t1; i += kSplitBlock) {
        const int32_t r = static_cast<int32_t>(token_row(ids, i, a.lo, a.lo + a.rows, a.padding_idx));
        if (r >= 0) atomicAdd(&cursor[r & (a.segments - 1)], 1);
    }
    __syncthreads();
    constexpr int kPer = kSegments / kSplitBlock;
    const int per = a.segments / kSplitBlock;      // 1 to kPer segments per thread
    int32_t n[kPer], total = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        n[k] = k < per ? cursor[t * per + k] : 0;
        total += n[k];
    }
    int32_t incl = total;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t up = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += up;
    }
    if (lane == kWave - 1) wave_total[wave] = incl;
    __syncthreads();
    int32_t run = incl - total;
#pragma unroll
    for (int k = 0; k < kSplitBlock / kWave; ++k) run += k < wave ? wave_total[k] : 0;
    int32_t* const offsets = a.offsets + static_cast<int64_t>(blockIdx.x) * (a.segments + 1);
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (k >= per) break;
        cursor[t * per + k] = run;
        offsets[t * per + k] = run;
        run += n[k];
    }
    if (t == kSplitBlock - 1) offsets[a.segments] = run;
    __syncthreads();
    for (int64_t i = t0 + t; i < t1; i += kSplitBlock) {
        const int32_t r = static_cast<int32_t>(token_row(ids, i, a.lo, a.lo + a.rows, a.padding_idx));
        if (r < 0) continue;
        const int64_t at = t0 + atomicAdd(&cursor[r & (a.segments - 1)], 1);
        a.token[at] = static_cast<int32_t>(i);
        a.row[at] = r >> a.shift;
    }
}

// One counter takes the lanes of a wavefront that share the first active lane's row in one atomic: a bucket of thousands of
// tokens is mostly such lanes.  Returns what the counter held, plus the lane's place among them.
__device__ inline int32_t count_up(int32_t* counters, int32_t row) {
    const int32_t first = __builtin_amdgcn_readfirstlane(row);
    const uint64_t same = __ballot(row == first);
    if (row != first) return atomicAdd(&counters[row], 1);
    const int32_t before = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(same >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(same), 0));
    int32_t base = 0;
    if (before == 0) base = atomicAdd(&counters[first], __popcll(same));
    return __builtin_amdgcn_readfirstlane(base) + before;
}

// ONE: without emb_bwd_split in front; each workgroup looks at all tokens and keeps its segment's in LDS.  Its hot rows go into slots
// of its own, for there is no launch in front that could clear a counter.
template <typename IdT, bool ONE>
__global__ __launch_bounds__(kBucketBlock) void emb_bwd_buckets(const IdT* __restrict__ ids, const SplitArgs a) {
    constexpr int kSegRows = ONE ? kOneRows : kSegmentRows;
    __shared__ int32_t counters[kSegRows];
    __shared__ int32_t upto[ONE ? 1 : kChunks + 1], from[ONE ? 1 : kChunks];   // tokens of this segment in the chunks below; where its own begin
    __shared__ uint16_t my_token[ONE ? kOneTokens : 1], my_row[ONE ? kOneTokens : 1];
    __shared__ int32_t my_tokens, my_hot;
    __shared__ int32_t wave_total[kBucketBlock / kWave], wave_base[kBucketBlock / kWave];
    __shared__ int32_t held[kHeldTokens];
    __shared__ uint16_t held_row[kHeldTokens];
    __shared__ int32_t long_begin[kLongRows], long_end[kLongRows], long_rows;
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
    const int32_t s = static_cast<int32_t>(blockIdx.x);
    if (t == 0) long_rows = 0;
    const int32_t rows = s < a.rows ? ((a.rows - 1 - s) >> a.shift) + 1 : 0;   // of this segment
    for (int i = t; i < rows; i += kBucketBlock) counters[i] = 0;
    int32_t tokens = 0, run = 0;                  // of this segment; of the segments below: where this one's stretch begins
    if constexpr (ONE) {
        if (t == 0) my_tokens = my_hot = 0;
        __syncthreads();
        int32_t lower = 0;
        constexpr int kEach = kOneTokens / kBucketBlock;
        int32_t r[kEach];
#pragma unroll
        for (int k = 0; k < kEach; ++k) {
            const int64_t i = t + k * kBucketBlock;
            r[k] = i < a.n_ids ? static_cast<int32_t>(token_row(ids, i, a.lo, a.lo + a.rows, a.padding_idx)) : -1;
        }
#pragma unroll
        for (int k = 0; k < kEach; ++k) {
            const int32_t segment = r[k] & (a.segments - 1);
            const bool mine = r[k] >= 0 && segment == s;
            lower += r[k] >= 0 && segment < s ? 1 : 0;
            const uint64_t all = __ballot(mine);
            if (all == 0) continue;                    // the same in all lanes
            const int32_t before = __popcll(all & ((1ull << lane) - 1));
            int32_t first = 0;
            if (lane == 0) first = atomicAdd(&my_tokens, __popcll(all));
            const int32_t at = __builtin_amdgcn_readfirstlane(first) + before;
            if (mine) my_token[at] = static_cast<uint16_t>(t + k * kBucketBlock), my_row[at] = static_cast<uint16_t>(r[k] >> a.shift);
        }
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) lower += __shfl_xor(lower, off, kWave);
        if (lane == kWave - 1) wave_base[wave] = lower;
        __syncthreads();
        tokens = my_tokens;
#pragma unroll
        for (int k = 0; k < kBucketBlock / kWave; ++k) run += wave_base[k];
    } else {
        // A thread per chunk.  The tokens of lower segments in all chunks are the place of this segment's stretch.
        static_assert(kChunks == kBucketBlock, "a thread per chunk");
        int32_t len = 0, lower = 0;
        if (t < a.chunks) {
            const int32_t* const o = a.offsets + static_cast<int64_t>(t) * (a.segments + 1) + s;
            lower = o[0];
            len = o[1] - lower;
            from[t] = lower;
        }
        int32_t incl = len, base = lower;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int32_t up = __shfl_up(incl, off, kWave);
            if (lane >= off) incl += up;
            base += __shfl_xor(base, off, kWave);
        }
        if (lane == kWave - 1) wave_total[wave] = incl, wave_base[wave] = base;
        __syncthreads();
        int32_t before = 0;
#pragma unroll
        for (int k = 0; k < kBucketBlock / kWave; ++k) {
            before += k < wave ? wave_total[k] : 0;
            tokens += wave_total[k];
            run += wave_base[k];
        }
        upto[t + 1] = before + incl;
        if (t == 0) upto[0] = 0;
        __syncthreads();
    }
    // Where this segment's token i < tokens is: in the chunk c with upto[c] <= i < upto[c + 1].
    auto place = [&](int32_t i) {
        int32_t c = 0;
#pragma unroll
        for (int32_t half = kChunks / 2; half > 0; half >>= 1)
            if (upto[c + half] <= i) c += half;
        return c * a.chunk_tokens + from[c] + (i - upto[c]);
    };
    auto look = [&](int32_t i, int32_t& row, int32_t& token) {
        if constexpr (ONE) {
            row = my_row[i], token = my_token[i];
        } else {
            const int64_t at = place(i);
            row = a.row[at], token = a.token[at];
        }
    };
    // The first kBucketBlock tokens, mostly all, stay in registers.
    int32_t row_first = -1, token_first = 0;
    if (t < tokens) {
        look(t, row_first, token_first);
        count_up(counters, row_first);
    }
    for (int32_t i = t + kBucketBlock; i < tokens; i += kBucketBlock) {
        int32_t row, token;
        look(i, row, token);
        count_up(counters, row);
    }
    __syncthreads();
    constexpr int kRows = kSegRows / kBucketBlock;
    const int per = (rows + kBucketBlock - 1) / kBucketBlock;   // consecutive rows of a thread
    int32_t n[kRows], begins[kRows], long_at[kRows], total = 0;
    const int32_t run_first = run;                              // where this segment's stretch begins
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        long_at[k] = -1, begins[k] = 0;
        n[k] = k < per && t * per + k < rows ? counters[t * per + k] : 0;
        total += n[k];
    }
    int32_t incl = total;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t up = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += up;
    }
    __syncthreads();                                            // wave_total has been read
    if (lane == kWave - 1) wave_total[wave] = incl;
    __syncthreads();
    run += incl - total;
#pragma unroll
    for (int k = 0; k < kBucketBlock / kWave; ++k) run += k < wave ? wave_total[k] : 0;
    Row* const meta = a.meta + static_cast<int64_t>(s) * a.segment_rows;
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        const int32_t r = t * per + k;
        if (k >= per || r >= rows) break;
        counters[r] = begins[k] = run;
        run += n[k];
        meta[r].count = n[k], meta[r].end = run;
        // Long rows from the front of the list, so that their workgroups start first; the others from its end.
        if constexpr (ONE) {
            if (n[k] > kRankTokens) long_at[k] = atomicAdd(&long_rows, 1);
            if (n[k] > a.hot_above)
                a.hot[hot_slots(run_first, s) + atomicAdd(&my_hot, 1)] = ((r << a.shift) + s) | (n[k] > kRankTokens ? kOrdered | kLong : tokens <= kHeldTokens ? kOrdered : 0);
        } else if (n[k] > kRankTokens) {
            if (a.n_ids <= kBitsPerWindow) long_at[k] = atomicAdd(&long_rows, 1);
            a.hot[atomicAdd(&a.totals[1], 1)] = ((r << a.shift) + s) | (a.n_ids <= kBitsPerWindow ? kOrdered : 0);
        } else if (n[k] > a.hot_above) {
            a.hot[a.hot_most - 1 - atomicAdd(&a.totals[0], 1)] = ((r << a.shift) + s) | (tokens <= kHeldTokens ? kOrdered : 0);
        }
    }
    __syncthreads();
    if constexpr (ONE) {   // the slots that are left
        const int32_t end = hot_slots(s + 1 < a.segments ? run_first + tokens : static_cast<int32_t>(a.n_ids), s + 1);
        for (int32_t i = hot_slots(run_first, s) + my_hot + t; i < end; i += kBucketBlock) a.hot[i] = -1;
    }
    // The buckets, in ascending order where that is cheap: the workgroups that share a hot row's columns need not each do it.
    const int32_t stretch = run_first;
    if (tokens <= kHeldTokens) {
        auto hold = [&](int32_t row, int32_t token) {
            const int32_t at = count_up(counters, row) - stretch;
            held[at] = token, held_row[at] = static_cast<uint16_t>(row);
        };
        if (row_first >= 0) hold(row_first, token_first);
        for (int32_t i = t + kBucketBlock; i < tokens; i += kBucketBlock) {
            int32_t row, token;
            look(i, row, token);
            hold(row, token);
        }
        __syncthreads();
        for (int32_t i = t; i < tokens; i += kBucketBlock) {   // a counter holds the end of its row now, which is where the next begins
            const int32_t r = held_row[i], begin = r ? counters[r - 1] - stretch : 0, end = counters[r] - stretch;
            int32_t to = i;
            if (end - begin > 1 && end - begin <= kRankTokens) {
                const int32_t mine = held[i];
                to = begin;
#pragma unroll 8
                for (int32_t j = begin; j < end; ++j) to += held[j] < mine ? 1 : 0;
            }
            a.bucket[stretch + to] = held[i];
        }
    } else {
        if (row_first >= 0) a.bucket[count_up(counters, row_first)] = token_first;
        for (int32_t i = t + kBucketBlock; i < tokens; i += kBucketBlock) {
            int32_t row, token;
            look(i, row, token);
            a.bucket[count_up(counters, row)] = token;
        }
    }
    __syncthreads();
    const int32_t all_long = long_rows;
    static_assert(kBitsPerWindow / (kRankTokens + 1) <= kLongRows, "no call has more long rows whose tokens fit the bits");
#pragma unroll
    for (int k = 0; k < kRows; ++k)
        if (long_at[k] >= 0) {
            long_begin[long_at[k]] = begins[k];
            long_end[long_at[k]] = begins[k] + n[k];
        }
    for (int32_t h = 0; h < all_long; ++h) {
        uint32_t* const bits = reinterpret_cast<uint32_t*>(counters);
        static_assert((ONE ? kOneTokens : kBitsPerWindow) <= 32 * kSegRows, "a bit per token number where the counters were");
        constexpr int kWords = kSegRows / kBucketBlock;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kWords; ++k) bits[t + k * kBucketBlock] = 0;
        __syncthreads();
        const int32_t begin = long_begin[h], end = long_end[h];
        for (int32_t i = begin + t; i < end; i += kBucketBlock) {
            const int32_t at = tokens <= kHeldTokens ? held[i - stretch] : a.bucket[i];
            atomicOr(&bits[at >> 5], 1u << (at & 31));
        }
        __syncthreads();
        uint32_t mine[kWords];
        int32_t sum = 0;
#pragma unroll
        for (int k = 0; k < kWords; ++k) {
            mine[k] = bits[t * kWords + k];
            sum += __popc(mine[k]);
        }
        int32_t up_to = sum;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int32_t up = __shfl_up(up_to, off, kWave);
            if (lane >= off) up_to += up;
        }
        if (lane == kWave - 1) wave_total[wave] = up_to;
        __syncthreads();
        int32_t rank = begin + up_to - sum;
#pragma unroll
        for (int k = 0; k < kBucketBlock / kWave; ++k) rank += k < wave ? wave_total[k] : 0;
#pragma unroll
        for (int k = 0; k < kWords; ++k)
            for (uint32_t w = mine[k]; w; w &= w - 1) a.bucket[rank++] = (t * kWords + k) * 32 + __ffs(w) - 1;
    }
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
    const Row* meta;
    const int32_t* bucket;
    const int32_t* hot;
    const int32_t* totals;
    int32_t shift, segment_rows;   // of the segments that `meta` is ordered by
    int32_t hot_most;              // entries the hot list has room for: long rows from its front, others from its end; 0: all
                                   // from its front, and the last row of the table on no list
    int64_t n_ids;
    int32_t nv;             // vectors of V elements per row; the last one is moved back to end with the row
    int32_t passes;         // groups of columns per row of the ordinary path
    int32_t rows_per_block;
    int32_t hot_above;      // rows of more tokens are hot
    int32_t hot_chunks;     // pieces of kHotBytes of a row
    int32_t scale_by_freq;
    int32_t slots;          // not 0: hot rows are in this many slots, some of them empty, and `totals` holds nothing
    __device__ Row of(int64_t row) const { return meta[(row & ((1 << shift) - 1)) * segment_rows + (row >> shift)]; }
};

// ---- hot rows ----
// A workgroup owns 64 bytes of columns of one row.  What takes time is the
// memory round trip, not the additions, so all threads fetch the pieces of the
// next two batches -- four lanes a token, 16 bytes a lane -- while one
// wavefront adds a batch in token order out of LDS, a column per lane: the sums stay strictly sequential per column with 512 tokens in
// flight in emb_bwd_hot (batches of 256), 256 in emb_bwd_sums (of 128).  (With 256 bytes of columns and batches of 64 tokens a row of
// 11000 tokens of 512 bytes took 370 us, in emb_bwd_hot 100; 483 tokens of 2 KiB 20 us and 9.  A wavefront
// that walks its columns alone keeps 32 tokens in flight in the same registers: 55 us.)
// The order of the tokens, where emb_bwd_buckets has not made it: up to 512 by counting the smaller ones, more through
// a bit per token number in LDS (16 KiB for a window of 131072 of them) that is
// read back in ascending order, kListTokens at a time.  The bits have LDS of their
// own: in the stage's they had to be set again, by a walk over the whole bucket,
// for every kListTokens (2^20 tokens of one row, 256 bytes each: 1267 ms, now 59).
constexpr int kHotBytes = 64;
constexpr int kListTokens = 1024;
constexpr int kWordsPerThread = kBitWords / kBlock;

// SHORT: no unordered bucket of more than kRankTokens tokens.
template <typename E, bool SHORT>
struct HotShared {
    static constexpr int kBatch = SHORT ? 128 : 256;   // tokens per batch
    static constexpr int kPitch = kBatch + 4;        // 16 floats apart for the four lanes that store a token: no two on one bank
    alignas(16) float column[kHotBytes / sizeof(typename E::word)][kPitch];   // a batch in fp32, column by column: the adding wavefront reads four tokens at once
    alignas(16) uint32_t bits[SHORT ? kRankTokens : kBitWords];   // a bit per token number, or the bucket being ordered
    int32_t list[SHORT ? kRankTokens : kListTokens];   // tokens in ascending order
    int32_t wave_total[kWavesPerBlock];
    int32_t found[SHORT ? kHotSlots : 1], slots[4][kWavesPerBlock];   // the entries of the slots, long rows first
};

// Adds the m tokens of the list (in LDS or in global memory) to the columns from col0 on, thread t's to column col0 + t; called by all
// threads.
template <typename E, bool SHORT>
__device__ inline void hot_accumulate(HotShared<E, SHORT>& sh, const ReduceArgs& a, const int32_t* list, int64_t col0, int m, float& acc) {
    typedef typename E::word W;
    constexpr int kBatch = HotShared<E, SHORT>::kBatch;
    constexpr int V = 16 / sizeof(W), kCols = kHotBytes / sizeof(W);
    constexpr int kLanesPerToken = kHotBytes / 16, kTokensPerLoad = kBlock / kLanesPerToken, kLoads = kBatch / kTokensPerLoad;
    const int t = threadIdx.x, part = t % kLanesPerToken, tok0 = t / kLanesPerToken;
    const int64_t col = col0 + part * V, left = a.dim - col;
    const W* const dy = static_cast<const W*>(a.dy) + col;
    Pack<W, V> piece[2][kLoads];
    int32_t token[kLoads];                           // of the batch that is fetched next
    auto look = [&](int base) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int i = base + u * kTokensPerLoad + tok0;
            token[u] = i < m ? list[i] : 0;
        }
    };
    auto fetch = [&](Pack<W, V> (&to)[kLoads], int base) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int i = base + u * kTokensPerLoad + tok0;
            if (i >= m || left <= 0) continue;
            const W* src = dy + static_cast<int64_t>(token[u]) * a.ld_dy;
            if (left >= V) {
                to[u] = load_pack<W, V>(src);
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) to[u].e[e] = e < left ? src[e] : W(0);
            }
        }
    };
    auto batch = [&](Pack<W, V> (&from)[kLoads], int base) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
#pragma unroll
            for (int e = 0; e < V; ++e) sh.column[part * V + e][u * kTokensPerLoad + tok0] = E::widen(from[u].e[e]);
        __syncthreads();
        if (base + 2 * kBatch < m) fetch(from, base + 2 * kBatch);
        if (base + 3 * kBatch < m) look(base + 3 * kBatch);
        if (t < kCols) {
            const int here = m - base < kBatch ? m - base : kBatch;
            const float* const mine = sh.column[t];
            int k = 0;
            for (; k + 32 <= here; k += 32) {
                float4 q[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) q[u] = *reinterpret_cast<const float4*>(&mine[k + 4 * u]);
#pragma unroll
                for (int u = 0; u < 8; ++u) acc += q[u].x, acc += q[u].y, acc += q[u].z, acc += q[u].w;
            }
            for (; k < here; ++k) acc += mine[k];
        }
        __syncthreads();
    };
    look(0);
    fetch(piece[0], 0);
    if (kBatch < m) {
        look(kBatch);
        fetch(piece[1], kBatch);
    }
    if (2 * kBatch < m) look(2 * kBatch);
    for (int base = 0; base < m; base += 2 * kBatch) {
        batch(piece[0], base);
        if (base + kBatch < m) batch(piece[1], base + kBatch);
    }
}

// Called by every thread of the workgroup with the same arguments.
template <typename E, bool SHORT>
__device__ inline void hot_row(HotShared<E, SHORT>& sh, const ReduceArgs& a, int64_t row, bool ordered, int chunk) {
    typedef typename E::word W;
    const Row meta = a.of(row);
    const int32_t n = meta.count;
    const int32_t* const bucket = a.bucket + (meta.end - n);
    const int t = threadIdx.x;
    const int64_t col0 = static_cast<int64_t>(chunk) * (kHotBytes / sizeof(W));
    float acc = 0.f;
    if (ordered) {
        hot_accumulate<E, SHORT>(sh, a, bucket, col0, n, acc);
    } else if (n <= kRankTokens) {
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
        hot_accumulate<E, SHORT>(sh, a, sh.list, col0, n, acc);
    } else if constexpr (!SHORT) {
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
                hot_accumulate<E, SHORT>(sh, a, sh.list, col0, here < kListTokens ? here : kListTokens, acc);
            }
        }
    }
    if (t < static_cast<int>(kHotBytes / sizeof(W)) && col0 + t < a.dim) {
        const float scale = (a.scale_by_freq && n > 1) ? 1.0f / static_cast<float>(n) : 1.0f;
        static_cast<W*>(a.dw)[row * a.ld_dw + col0 + t] = E::round(acc * scale);
    }
    __syncthreads();                                 // the list is rewritten by the workgroup's next row
}

// Item after item by `blocks` workgroups.
template <typename E, bool SHORT>
__device__ inline void hot_rows(HotShared<E, SHORT>& sh, const ReduceArgs& a, int32_t block, int32_t blocks) {
    int32_t listed, more = 0;
    const bool slots = SHORT && a.slots != 0;
    if (slots) {
        static_assert(kHotSlots == 2 * kBlock, "two slots a thread");
        const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
        const int32_t e0 = t < a.slots ? a.hot[t] : -1, e1 = t + kBlock < a.slots ? a.hot[t + kBlock] : -1;
        const uint64_t in[4] = {__ballot(e0 >= 0 && (e0 & kLong)), __ballot(e1 >= 0 && (e1 & kLong)), __ballot(e0 >= 0 && !(e0 & kLong)),
                                __ballot(e1 >= 0 && !(e1 & kLong))};
        if (lane < 4) sh.slots[lane][wave] = __popcll(lane == 0 ? in[0] : lane == 1 ? in[1] : lane == 2 ? in[2] : in[3]);
        __syncthreads();
        listed = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            int32_t at = listed;
#pragma unroll
            for (int k = 0; k < kWavesPerBlock; ++k) {
                at += k < wave ? sh.slots[q][k] : 0;
                listed += sh.slots[q][k];
            }
            if ((in[q] >> lane) & 1) sh.found[at + __popcll(in[q] & ((1ull << lane) - 1))] = (q & 1 ? e1 : e0) & ~kLong;
        }
        __syncthreads();
    } else {
        listed = a.totals[1];
        more = a.hot_most ? a.totals[0] : a.of(a.rows - 1).count > a.hot_above ? 1 : 0;
    }
    const int32_t items = (listed + more) * a.hot_chunks;
    for (int32_t item = block; item < items; item += blocks) {
        const int32_t which = item / a.hot_chunks;
        const int32_t entry = slots ? sh.found[which] : which < listed ? a.hot[which] : a.hot_most ? a.hot[a.hot_most - 1 - (which - listed)] : static_cast<int32_t>(a.rows) - 1;
        const bool ordered = a.hot_most && (entry & kOrdered);
        hot_row<E, SHORT>(sh, a, ordered ? entry & ~kOrdered : entry, ordered, item - which * a.hot_chunks);
    }
}

// A launch of its own where a hot row's bucket may have to be ordered through the bits: with their LDS the ordinary rows, which
// live on many wavefronts, took 64 us instead of 50 for [16032,4096] bf16.
template <typename E>
__global__ __launch_bounds__(kBlock) void emb_bwd_hot(const ReduceArgs a) {
    __shared__ HotShared<E, false> sh;
    hot_rows<E, false>(sh, a, static_cast<int32_t>(blockIdx.x), static_cast<int32_t>(gridDim.x));
}

// ---- ordinary rows ----
// V: elements per vector (16 bytes, or 1 for rows shorter than that).  LPR lanes
// share a row (32: two rows per wavefront, for rows of at most 32 vectors), CPW
// vectors per lane and pass.  Buckets (of at most kHotAbove tokens) are ordered in
// registers: lane i holds one token, counts the smaller ones (its rank) and sends
// it to the lane of that number (lanes without a token send theirs, larger than
// any, to the lane behind the last).
template <typename E, int V, int LPR, int CPW>
__device__ __forceinline__ void ordinary_rows(const ReduceArgs& a, uint32_t block) {
    typedef typename E::word W;
    constexpr int kGroups = kWave / LPR;
    const int lane = threadIdx.x & (kWave - 1), g = lane / LPR, gl = lane % LPR;
    const int64_t row0 = static_cast<int64_t>(block) * a.rows_per_block;
    const int items = a.rows_per_block / kGroups * a.passes;
    const W* const dy = static_cast<const W*>(a.dy);
    for (int item = threadIdx.x / kWave; item < items; item += kWavesPerBlock) {
        const int q = item / a.passes, pass = item - q * a.passes;
        const int64_t row = row0 + q * kGroups + g;
        const bool real = row < a.rows;
        const Row meta = real ? a.of(row) : Row{0, 0};
        int32_t n = meta.count;
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
            int32_t tok = gl < n ? a.bucket[meta.end - n + gl] : 0x7FFFFFFF;
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

template <typename E, int V, int LPR, int CPW>
__global__ __launch_bounds__(kBlock, 8) void emb_bwd_reduce(const ReduceArgs a) {
    ordinary_rows<E, V, LPR, CPW>(a, blockIdx.x);
}

// Hot and ordinary rows in one launch, the hot ones first: two launches wait for each other, the hot rows' mostly for memory and the
// others' for their stores.  Batches of 128 tokens and no bits leave room for six wavefronts a SIMD (with batches of 256, four: [16032,
// 4096] bf16 of 131072 tokens, of which 16384 hit, 58.1 us, here 51.7, two launches 53.6).  The whole gradient, two launches -> one:
// 8192 tokens as in text, [50304, 512] fp32 39.8 -> 33.3 us; 32768, 62.6 -> 49.8; 32768, [65000, 4096] bf16 251 -> 184; 4096, [16032,
// 4096] 49.8 -> 35.8; 131072, [16032, 512] 146 -> 142; uniform: 16384, [65000, 4096] 111 -> 106, 65536, [16032, 4096] 140 -> 135.
template <typename E, int V, int LPR, int CPW>
__global__ __launch_bounds__(kBlock, 6) void emb_bwd_sums(const ReduceArgs a, int32_t hot_blocks) {
    __shared__ HotShared<E, true> sh;
    if (static_cast<int32_t>(blockIdx.x) < hot_blocks) hot_rows<E, true>(sh, a, static_cast<int32_t>(blockIdx.x), hot_blocks);
    else ordinary_rows<E, V, LPR, CPW>(a, blockIdx.x - hot_blocks);
}

template <typename E, int V>
void launch_reduce(ReduceArgs a, bool together, uint32_t hot_blocks, hipStream_t s) {
    a.nv = static_cast<int32_t>((a.dim + V - 1) / V);
    auto go = [&](auto kernel, auto with_hot, int lpr, int cpw) {
        a.passes = (a.nv + lpr * cpw - 1) / (lpr * cpw);
        // One row per workgroup when a row has work for three or four wavefronts, else as many rows as fill them.
        a.rows_per_block = a.passes >= 3 ? 1 : (kWave / lpr) * (kWavesPerBlock / a.passes);
        const int64_t blocks = (a.rows + a.rows_per_block - 1) / a.rows_per_block;
        if (together && hot_blocks > 0) {
            hipLaunchKernelGGL(with_hot, dim3(static_cast<uint32_t>(blocks + hot_blocks)), dim3(kBlock), 0, s, a, static_cast<int32_t>(hot_blocks));
        } else {
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kBlock), 0, s, a);
        }
    };
    if (a.nv <= 32)
        go(emb_bwd_reduce<E, V, 32, 1>, emb_bwd_sums<E, V, 32, 1>, 32, 1);
    else if (a.nv <= 64)
        go(emb_bwd_reduce<E, V, 64, 1>, emb_bwd_sums<E, V, 64, 1>, 64, 1);
    else
        go(emb_bwd_reduce<E, V, 64, 2>, emb_bwd_sums<E, V, 64, 2>, 64, 2);
}

template <typename E>
void launch_reduce_any(const ReduceArgs& a, uint32_t hot_blocks, hipStream_t s) {
    constexpr int V = 16 / sizeof(typename E::word);
    // One launch where emb_bwd_buckets has put all long rows in order (slots are read by emb_bwd_sums alone, and only of so few tokens).
    static_assert(kOneTokens <= kBitsPerWindow, "slots are left by emb_bwd_buckets");
    const bool together = a.hot_most && a.n_ids <= kBitsPerWindow;
    // Few tokens have few hot rows, and workgroups that find none keep the ordinary rows waiting (8192 tokens as in text, [50304, 512]
    // fp32: 256 workgroups 33.3 us, 2048 35.0; 32768: 69.6 and 49.8).
    if (a.slots) hot_blocks = std::min<uint32_t>(hot_blocks, 256);
    if (hot_blocks > 0 && !together) hipLaunchKernelGGL(emb_bwd_hot<E>, dim3(hot_blocks), dim3(kBlock), 0, s, a);
    if (a.dim >= V)
        launch_reduce<E, V>(a, together, hot_blocks, s);
    else
        launch_reduce<E, 1>(a, together, hot_blocks, s);
}

// Chunks, segments and workspace (elems int32; 0: too many rows) of the bucketing in two launches.
struct Split {
    int64_t elems, chunk_tokens;
    int shift, segment_rows, chunks;
};

Split plan_split(int64_t n_ids, int64_t rows) {
    Split p{};
    if (n_ids < 1 || rows > static_cast<int64_t>(kSegments) * kSegmentRows) return p;
    p.shift = 8;
    while ((rows - 1) >> p.shift >= kSegmentRows) ++p.shift;
    p.segment_rows = static_cast<int>(((rows - 1) >> p.shift) + 1);
    p.chunk_tokens = (n_ids + kChunks - 1) / kChunks;
    if (p.chunk_tokens < 1024) p.chunk_tokens = 1024;
    p.chunks = static_cast<int>((n_ids + p.chunk_tokens - 1) / p.chunk_tokens);
    const int64_t segments = 1ll << p.shift;
    p.elems = 2 * segments * p.segment_rows + 2 + 3 * n_ids + p.chunks * (segments + 1) + hot_slots(static_cast<int32_t>(n_ids), static_cast<int32_t>(segments));
    return p;
}

template <typename IdT>
int run(const void* dy, int dtype, int64_t dim, int64_t ld_dy, const IdT* ids, int64_t n_ids, int64_t lo, int64_t hi,
        int64_t padding_idx, int scale_by_freq, void* dw, int64_t ld_dw, int32_t* ws, int64_t ws_elems, hipStream_t s) {
    const int64_t rows = hi - lo;
    const int es = dtype == DDL_DT_F32 ? 4 : 2;
    ReduceArgs a{};
    a.dy = dy, a.dw = dw, a.dim = dim, a.ld_dy = ld_dy, a.ld_dw = ld_dw, a.rows = rows, a.n_ids = n_ids;
    a.scale_by_freq = scale_by_freq;
    a.hot_above = kHotAbove;
    const int64_t most_hot = std::min(rows, n_ids / (a.hot_above + 1));
    a.hot_chunks = static_cast<int32_t>((dim * es + kHotBytes - 1) / kHotBytes);
    const uint32_t hot_blocks = static_cast<uint32_t>(std::min<int64_t>(most_hot * a.hot_chunks, 2048));
    const Split split = plan_split(n_ids, rows);
    if (split.elems && split.elems <= ws_elems) {
        SplitArgs b{};
        b.n_ids = n_ids, b.lo = lo, b.padding_idx = padding_idx, b.chunk_tokens = split.chunk_tokens;
        b.rows = static_cast<int32_t>(rows), b.segments = 1 << split.shift, b.shift = split.shift;
        b.hot_most = static_cast<int32_t>(n_ids / (kHotAbove + 1) + 1);
        b.segment_rows = split.segment_rows, b.chunks = split.chunks, b.hot_above = a.hot_above;
        b.meta = reinterpret_cast<Row*>(ws);
        b.totals = ws + 2 * static_cast<int64_t>(b.segments) * b.segment_rows;
        b.bucket = b.totals + 2;
        b.token = b.bucket + n_ids;
        b.row = b.token + n_ids;
        b.offsets = b.row + n_ids;
        b.hot = b.offsets + static_cast<int64_t>(b.chunks) * (b.segments + 1);
        a.meta = b.meta, a.bucket = b.bucket, a.hot = b.hot, a.totals = b.totals;
        a.shift = b.shift, a.segment_rows = b.segment_rows, a.hot_most = b.hot_most;
        if (n_ids <= kOneTokens && b.segments == 256 && b.segment_rows <= kOneRows) {
            a.slots = hot_slots(static_cast<int32_t>(n_ids), b.segments);
            hipLaunchKernelGGL((emb_bwd_buckets<IdT, true>), dim3(static_cast<uint32_t>(b.segments)), dim3(kBucketBlock), 0, s, ids, b);
        } else {
            hipLaunchKernelGGL((emb_bwd_split<IdT>), dim3(static_cast<uint32_t>(b.chunks)), dim3(kSplitBlock), 0, s, ids, b);
            hipLaunchKernelGGL((emb_bwd_buckets<IdT, false>), dim3(static_cast<uint32_t>(b.segments)), dim3(kBucketBlock), 0, s, ids, b);
        }
    } else {
        // 3 rows + 1 + n_ids integers: the hot list has at most rows - 1 entries
        Row* const meta = reinterpret_cast<Row*>(ws);           // [rows]
        int32_t* const totals = ws + 2 * rows;                  // [2]
        int32_t* const bucket = totals + 2;                     // [n_ids]
        int32_t* const hot = bucket + n_ids;                    // [rows - 1]
        a.meta = meta, a.bucket = bucket, a.hot = hot, a.totals = totals;
        a.shift = 0, a.segment_rows = 0, a.hot_most = 0;
        auto grid = [](int64_t n) { return dim3(static_cast<uint32_t>((n + kBlock - 1) / kBlock)); };
        hipLaunchKernelGGL(emb_bwd_clear, grid(std::max<int64_t>(rows, 2)), dim3(kBlock), 0, s, meta, rows, totals);
        if (n_ids > 0) {
            hipLaunchKernelGGL((emb_bwd_count<IdT>), grid(n_ids), dim3(kBlock), 0, s, ids, n_ids, lo, hi, padding_idx, meta);
            hipLaunchKernelGGL(emb_bwd_place, grid((rows + kPlaceRows - 1) / kPlaceRows), dim3(kBlock), 0, s, meta, rows, a.hot_above, hot, totals);
            hipLaunchKernelGGL((emb_bwd_fill<IdT>), grid(n_ids), dim3(kBlock), 0, s, ids, n_ids, lo, hi, padding_idx, meta, bucket);
        }
    }
    if (dtype == DDL_DT_F16)
        launch_reduce_any<F16>(a, hot_blocks, s);
    else if (dtype == DDL_DT_BF16)
        launch_reduce_any<Bf16>(a, hot_blocks, s);
    else
        launch_reduce_any<F32>(a, hot_blocks, s);
    return check_launch("embedding backward");
}

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

extern "C" int64_t ddl_embedding_backward_workspace(int64_t n_ids, int64_t rows) {
    using namespace ddl;
    if (n_ids < 0 || rows < 0 || n_ids > 0x7FFFFFFFll || rows > 0x3FFFFFFFll) return 0;
    return std::max(plan_split(n_ids, rows).elems, 3 * rows + 1 + n_ids);
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
                   ld_dw, workspace, workspace_elems, s);
    return run(dy, dtype, dim, ld_dy, static_cast<const int32_t*>(ids), n_ids, lo, hi, padding_idx, scale_grad_by_freq != 0, dweight, ld_dw,
               workspace, workspace_elems, s);
}
