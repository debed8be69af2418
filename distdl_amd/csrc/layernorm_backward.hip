// Backward of the DistributedLayerNorm shard: what autograd derives from
// the reference's forward (nn/layernorm.py:230-247, 295-309)
//
//   mean = allreduce(local mean) / P        var = allreduce(local mean((x-mean)^2)) / P
//   xhat = (x - mean) rstd                  y = gamma xhat + beta
//
// Every element of worker p enters mean and var with weight a_p = 1 / (P n_p)
// (n_p = columns held by p; the weights of a row add up to 1), which gives
//
//   g    = dy gamma
//   S1   = sum over the whole row of g           S2 = sum over the whole row of g xhat
//   dx   = rstd (g - a_p (S1 + xhat S2))
//   dgamma[c] = sum over rows of dy xhat         dbeta[c] = sum over rows of dy
//
// S1 and S2 span all workers of the row, so the work is split like the forward:
//   ln_bwd_partial   local {sum g, sum g xhat} per row      (one read of dy, x)
//   -- the caller gathers the pairs of the P workers --
//   ln_bwd_input     sums the gathered pairs, writes dx      (one read of dy, x)
//   ln_bwd_params    column sums over the local rows, in row splits through a
//                    workspace, for dgamma and dbeta
// One wavefront owns a row and strides over its columns (four elements at a time
// when the row is aligned); nothing is kept between passes, so rows of any length
// work.  Callers that want dx and the parameter gradients get fewer passes:
//   ln_bwd_partial_cols   row sums, column sums and (rows held whole, or the other
//                         workers' sums in memory) dx in one pass, a wavefront per
//                         row of at most 1024 columns
//   ln_bwd_block_rows     the same with a workgroup per longer row
// dy, x, gamma, dx, dgamma and dbeta are float, bf16 or fp16 (one type per
// call); the arithmetic, the saved mean and rstd, the row sums and the workspace
// are fp32.
#include "ln_elements.h"

namespace ddl {
namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kStrip = 64;     // columns per workgroup of the parameter kernel

constexpr int kAhead = 4;   // pieces of a row that a lane requests together

// Four elements of dy, x and gamma.  ANY: at any address.
template <typename T, bool ANY>
struct BwdPiece {
    float4 d, v, g;
    __device__ void load(const T* dy, const T* x, const T* gamma, int64_t c) {
        d = load_piece<ANY>(dy + c);
        v = load_piece<ANY>(x + c);
        g = gamma ? load_piece<ANY>(gamma + c) : make_float4(1.f, 1.f, 1.f, 1.f);
    }
};

// Column at which the piece from `c` on is fetched.  ANY: the last piece of a row of four columns and more ends with the
// row, and its first elements are those of the piece in front of it once more: left out of sums, written twice.  (A branch
// for the end of a row keeps the loads of the other pieces from being in flight.)
template <bool ANY, typename I>
__device__ inline I piece_column(I c, I cols) {
    return ANY && c + 4 > cols ? cols - 4 : c;
}

// The piece without the elements that the one in front of it has.
template <bool ANY>
__device__ inline float4 own_elements(float4 d, int again) {
    if (ANY && again > 0) {
        d.x = 0.f;
        if (again > 1) d.y = 0.f;
        if (again > 2) d.z = 0.f;
    }
    return d;
}

// ANY: rows of any length, pitch and address ([5461, 6143] bf16 81 us element by element, here 26; ln_bwd_input 68, here 36).
template <typename T, bool ANY>
__global__ __launch_bounds__(kBlock) void ln_bwd_partial(const T* __restrict__ dy, const T* __restrict__ x, int64_t rows,
                                                         int64_t cols, int64_t ld_dy, int64_t ld_x,
                                                         const float* __restrict__ mean, const float* __restrict__ rstd,
                                                         const T* __restrict__ gamma, float* __restrict__ sums) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t r = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + threadIdx.x / kWave;
    if (r >= rows) return;
    const float m = mean[r], rs = rstd[r];
    const T* dyr = dy + r * ld_dy;
    const T* xr = x + r * ld_x;
    float s1 = 0.f, s2 = 0.f;
    if (ANY && cols < 4) {
        if (lane < cols) {
            s1 = load1(dyr + lane) * (gamma ? load1(gamma + lane) : 1.f);
            s2 = s1 * ((load1(xr + lane) - m) * rs);
        }
    } else {
        for (int64_t first = lane * 4; first < cols; first += kAhead * kWave * 4) {
            BwdPiece<T, ANY> p[kAhead];
#pragma unroll
            for (int k = 0; k < kAhead; ++k)
                if (first + k * (kWave * 4) < cols) p[k].load(dyr, xr, gamma, piece_column<ANY>(first + k * (kWave * 4), cols));
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                const int64_t c = first + k * (kWave * 4);
                if (c >= cols) break;
                const float4 d = own_elements<ANY>(p[k].d, static_cast<int>(c - piece_column<ANY>(c, cols))), v = p[k].v, g = p[k].g;
                const float g0 = d.x * g.x, g1 = d.y * g.y, g2 = d.z * g.z, g3 = d.w * g.w;
                s1 += (g0 + g1) + (g2 + g3);
                s2 += (g0 * ((v.x - m) * rs) + g1 * ((v.y - m) * rs)) + (g2 * ((v.z - m) * rs) + g3 * ((v.w - m) * rs));
            }
        }
    }
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    if (lane == 0) reinterpret_cast<float2*>(sums)[r] = make_float2(s1, s2);
}

// One element of dx = rstd (g - (S1 + xhat S2)), S already times a_p.  Every
// kernel that writes dx goes through this one sequence of roundings (no
// contraction left to the compiler), so they agree bit for bit.
__device__ inline float dx_value(float dyv, float gv, float xv, float m, float rs, float S1, float S2) {
#pragma clang fp contract(off)
    const float h = (xv - m) * rs;
    const float t = __builtin_fmaf(h, S2, S1);
    const float q = dyv * gv - t;
    return rs * q;
}

template <typename T, bool ANY>
__device__ inline void ln_bwd_input_body(uint32_t block, const T* __restrict__ dy, const T* __restrict__ x, int64_t rows,
                                         int64_t cols, int64_t ld_dy, int64_t ld_x, const float* __restrict__ mean,
                                         const float* __restrict__ rstd, const T* __restrict__ gamma,
                                         const float* __restrict__ part_sums, int nparts, float weight, T* __restrict__ dx,
                                         int64_t ld_dx) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t r = static_cast<int64_t>(block) * kWavesPerBlock + threadIdx.x / kWave;
    if (r >= rows) return;
    // the pairs of all workers of this row, one worker per lane (and round)
    float p1 = 0.f, p2 = 0.f;
    for (int p = lane; p < nparts; p += kWave) {
        const float2 s = reinterpret_cast<const float2*>(part_sums)[static_cast<int64_t>(p) * rows + r];
        p1 += s.x;
        p2 += s.y;
    }
    const float m = mean[r], rs = rstd[r];
    const T* dyr = dy + r * ld_dy;
    const T* xr = x + r * ld_x;
    T* dxr = dx + r * ld_dx;
    // The first kAhead pieces of the row are requested before the sums are
    // reduced: the reduction waits for the gathered pairs, and the row should
    // not wait behind it (one memory round trip instead of two for rows of up
    // to 1024 columns).
    // Element by element where a row is shorter than a piece, and in place, where the last piece would start on elements that
    // have been stored.
    const bool by_element = ANY && (cols < 4 || dx == dy || dx == x);
    BwdPiece<T, ANY> p[kAhead];
    auto fetch = [&](int64_t first) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k)
            if (first + k * (kWave * 4) < cols) p[k].load(dyr, xr, gamma, piece_column<ANY>(first + k * (kWave * 4), cols));
    };
    int64_t first = lane * 4;
    if (!by_element) fetch(first);
    const float S1 = wave_sum(p1) * weight, S2 = wave_sum(p2) * weight;   // already times a_p
    if (by_element) {
        for (int64_t c = lane; c < cols; c += kWave) store1(dxr + c, dx_value(load1(dyr + c), gamma ? load1(gamma + c) : 1.f, load1(xr + c), m, rs, S1, S2));
        return;
    }
    while (true) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            const int64_t c = first + k * (kWave * 4);
            if (c < cols) {
                float4 o;
                o.x = dx_value(p[k].d.x, p[k].g.x, p[k].v.x, m, rs, S1, S2);
                o.y = dx_value(p[k].d.y, p[k].g.y, p[k].v.y, m, rs, S1, S2);
                o.z = dx_value(p[k].d.z, p[k].g.z, p[k].v.z, m, rs, S1, S2);
                o.w = dx_value(p[k].d.w, p[k].g.w, p[k].v.w, m, rs, S1, S2);
                store_piece<ANY>(dxr + piece_column<ANY>(c, cols), o);   // dx is not read again here: streaming store
            }
        }
        first += kAhead * kWave * 4;
        if (first >= cols) break;
        fetch(first);
    }
}

template <typename T, bool ANY>
__global__ __launch_bounds__(kBlock) void ln_bwd_input(const T* __restrict__ dy, const T* __restrict__ x, int64_t rows,
                                                       int64_t cols, int64_t ld_dy, int64_t ld_x,
                                                       const float* __restrict__ mean, const float* __restrict__ rstd,
                                                       const T* __restrict__ gamma, const float* __restrict__ part_sums,
                                                       int nparts, float weight, T* __restrict__ dx, int64_t ld_dx) {
    ln_bwd_input_body<T, ANY>(blockIdx.x, dy, x, rows, cols, ld_dy, ld_x, mean, rstd, gamma, part_sums, nparts, weight, dx, ld_dx);
}

// Workgroup (strip, split): rows [split * rows_per_split, ...) of a 64-column
// strip; lane group t / 64 takes every fourth row, thread t % 64 one column.
// partial[split, 0, c] = sum dy xhat, partial[split, 1, c] = sum dy.
template <typename T>
__global__ __launch_bounds__(kBlock) void ln_bwd_params_partial(const T* __restrict__ dy, const T* __restrict__ x,
                                                                int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                                                const float* __restrict__ mean, const float* __restrict__ rstd,
                                                                int64_t rows_per_split, float* __restrict__ partial, int strips) {
    __shared__ float fold[2][kWavesPerBlock][kStrip];
    const int split = blockIdx.x / strips, strip = blockIdx.x - split * strips;
    const int g = threadIdx.x / kStrip, t = threadIdx.x % kStrip;
    const int64_t c = static_cast<int64_t>(strip) * kStrip + t;
    const int64_t r_begin = split * rows_per_split;
    const int64_t r_end = r_begin + rows_per_split < rows ? r_begin + rows_per_split : rows;
    float a = 0.f, b = 0.f;
    if (c < cols) {
        for (int64_t r = r_begin + g; r < r_end; r += kWavesPerBlock) {
            const float d = load1(dy + r * ld_dy + c);
            a += d * ((load1(x + r * ld_x + c) - mean[r]) * rstd[r]);
            b += d;
        }
    }
    fold[0][g][t] = a;
    fold[1][g][t] = b;
    __syncthreads();
    if (threadIdx.x < 2 * kStrip) {
        const int which = threadIdx.x / kStrip;
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < kWavesPerBlock; ++k) s += fold[which][k][t];
        if (c < cols) partial[(static_cast<int64_t>(split) * 2 + which) * cols + c] = s;
    }
}

// Workgroup per 64-column strip: lane group g = t / 64 adds the splits g, g+4,
// ... of column t % 64 (independent loads, kInFlight of them requested together:
// many when this is all a kernel does, few when it shares its registers with
// the dx pass), LDS folds the four
// groups.
template <typename T, int kInFlight>
__device__ inline void ln_bwd_params_final_body(uint32_t block, const float* __restrict__ partial, int64_t cols, int splits,
                                                T* __restrict__ dgamma, T* __restrict__ dbeta) {
    __shared__ float fold[2][kWavesPerBlock][kStrip];
    const int g = threadIdx.x / kStrip, t = threadIdx.x % kStrip;
    const int64_t c = static_cast<int64_t>(block) * kStrip + t;
    float a = 0.f, b = 0.f;
    if (c < cols) {
        // Eight splits at a time, pairwise, whatever is in flight: a chain of 64 additions lost half as much again to rounding
        // ([3000, 2048] fp32 in 256 splits), and both callers add in the same order.
        auto fetch = [&](int k, float (&va)[8], float (&vb)[8]) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                va[u] = partial[(static_cast<int64_t>(k + u * kWavesPerBlock) * 2) * cols + c];
                vb[u] = partial[(static_cast<int64_t>(k + u * kWavesPerBlock) * 2 + 1) * cols + c];
            }
        };
        auto eight = [](const float (&v)[8]) { return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])); };
        constexpr int kEights = kInFlight / 8;
        int k = g;
        for (; k + (kInFlight - 1) * kWavesPerBlock < splits; k += kInFlight * kWavesPerBlock) {
            float va[kEights][8], vb[kEights][8];
#pragma unroll
            for (int e = 0; e < kEights; ++e) fetch(k + e * 8 * kWavesPerBlock, va[e], vb[e]);
#pragma unroll
            for (int e = 0; e < kEights; ++e) {
                a += eight(va[e]);
                b += eight(vb[e]);
            }
        }
        for (; k + 7 * kWavesPerBlock < splits; k += 8 * kWavesPerBlock) {
            float va[8], vb[8];
            fetch(k, va, vb);
            a += eight(va);
            b += eight(vb);
        }
        if (k < splits) {   // the last one to seven
            float va[8], vb[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int q = k + u * kWavesPerBlock;
                va[u] = q < splits ? partial[(static_cast<int64_t>(q) * 2) * cols + c] : 0.f;
                vb[u] = q < splits ? partial[(static_cast<int64_t>(q) * 2 + 1) * cols + c] : 0.f;
            }
            a += eight(va);
            b += eight(vb);
        }
    }
    fold[0][g][t] = a;
    fold[1][g][t] = b;
    __syncthreads();
    if (threadIdx.x < 2 * kStrip && c < cols) {
        const int which = threadIdx.x / kStrip;
        static_assert(kWavesPerBlock == 4, "four lane groups");
        const float s = (fold[which][0][t] + fold[which][1][t]) + (fold[which][2][t] + fold[which][3][t]);
        T* out = which == 0 ? dgamma : dbeta;
        if (out) store1(out + c, s);
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void ln_bwd_params_final(const float* __restrict__ partial, int64_t cols, int splits,
                                                              T* __restrict__ dgamma, T* __restrict__ dbeta) {
    ln_bwd_params_final_body<T, 32>(blockIdx.x, partial, cols, splits, dgamma, dbeta);
}

// dx and the final parameter sums in one launch: the first final_blocks
// workgroups (one per 64-column strip) add up the partial column sums -- a chain
// of dependent loads, so they start first -- and the rest write dx.  The two
// parts are independent.
template <typename T, bool ANY>
__global__ __launch_bounds__(kBlock) void ln_bwd_input_final(const T* __restrict__ dy, const T* __restrict__ x, int64_t rows,
                                                             int64_t cols, int64_t ld_dy, int64_t ld_x,
                                                             const float* __restrict__ mean, const float* __restrict__ rstd,
                                                             const T* __restrict__ gamma, const float* __restrict__ part_sums,
                                                             int nparts, float weight, T* __restrict__ dx, int64_t ld_dx,
                                                             uint32_t final_blocks, const float* __restrict__ partial, int splits,
                                                             T* __restrict__ dgamma, T* __restrict__ dbeta) {
    if (blockIdx.x < final_blocks)
        ln_bwd_params_final_body<T, 8>(blockIdx.x, partial, cols, splits, dgamma, dbeta);
    else
        ln_bwd_input_body<T, ANY>(blockIdx.x - final_blocks, dy, x, rows, cols, ld_dy, ld_x, mean, rstd, gamma, part_sums, nparts,
                               weight, dx, ld_dx);
}

constexpr int kFusedBlock = 512;   // eight wavefronts: a split of 32 rows is one round of four rows per wavefront
constexpr int kFusedWaves = kFusedBlock / kWave;

// What ln_bwd_partial_cols<.., true> needs beyond the sums: the other workers'
// row sums (already in memory), this worker's place among them, and where dx goes.
struct DxArgs {
    const float* part_sums;   // [nparts][rows][2]; slot my_part is not read
    int nparts, my_part;
    float weight;
    void* dx;
    int64_t ld_dx;
};

// Row sums {sum g, sum g xhat} and the partial column sums of a row split in one
// pass over dy and x: workgroup = split, its wavefronts take every eighth row
// and each lane keeps the columns (lane + 64 k) * 4 .. + 3, k < NV, in registers.
// partial has the layout of ln_bwd_params_partial.  WITH_DX: the sums of the
// whole row are complete once this worker's are (it holds the row whole, or the
// other workers' pairs are in memory), so dx is written in the same pass, from
// the registers that hold the row.  ANY: rows of at least four columns, of any length, pitch and address.
template <typename T, int NV, bool WITH_DX, bool ANY>
__global__ __launch_bounds__(kFusedBlock) void ln_bwd_partial_cols(const T* __restrict__ dy, const T* __restrict__ x, int64_t rows,
                                                              int64_t cols, int64_t ld_dy, int64_t ld_x,
                                                              const float* __restrict__ mean, const float* __restrict__ rstd,
                                                              const T* __restrict__ gamma, float* __restrict__ sums,
                                                              int64_t rows_per_split, float* __restrict__ partial, const DxArgs dxa) {
#pragma clang fp contract(off)   // both instantiations round alike: sums, column sums and dx do not depend on WITH_DX
    __shared__ float fold[2][kFusedWaves][NV * kWave * 4];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int nv = static_cast<int>((cols + 3) >> 2), n = static_cast<int>(cols);
    const int64_t r_begin = static_cast<int64_t>(blockIdx.x) * rows_per_split;
    const int64_t r_end = r_begin + rows_per_split < rows ? r_begin + rows_per_split : rows;
    float4 g[NV], ca[NV], cb[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c = lane + k * kWave;
        g[k] = make_float4(1.f, 1.f, 1.f, 1.f);
        if (gamma && c < nv) g[k] = load_piece<ANY>(gamma + piece_column<ANY>(4 * c, n));
        ca[k] = cb[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    constexpr int RU = NV <= 2 ? 4 : 2;   // rows whose loads are in flight together
    for (int64_t r0 = r_begin + wave; r0 < r_end; r0 += kFusedWaves * RU) {
        float m[RU], rs[RU];
        float4 d[RU][NV], v[RU][NV];
        float2 peer[RU];   // WITH_DX: the pair of worker `lane` for this row, requested together with the row
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const int64_t r = r0 + u * kFusedWaves;
            const bool on = r < r_end;
            m[u] = on ? mean[r] : 0.f;
            rs[u] = on ? rstd[r] : 0.f;
            peer[u] = make_float2(0.f, 0.f);
            if (WITH_DX && on && lane < dxa.nparts && lane != dxa.my_part)
                peer[u] = reinterpret_cast<const float2*>(dxa.part_sums)[static_cast<int64_t>(lane) * rows + r];
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int c = lane + k * kWave;
                d[u][k] = v[u][k] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (on && c < nv) {
                    d[u][k] = load_piece<ANY>(dy + r * ld_dy + piece_column<ANY>(4 * c, n));
                    v[u][k] = load_piece<ANY>(x + r * ld_x + piece_column<ANY>(4 * c, n));
                }
            }
        }
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const int64_t r = r0 + u * kFusedWaves;
            if (r >= r_end) break;                              // wave-uniform
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                // columns past the row hold zeros in d, so they add nothing
                const float4 dd = own_elements<ANY>(d[u][k], 4 * (lane + k * kWave) - piece_column<ANY>(4 * (lane + k * kWave), n)), vv = v[u][k];
                const float h0 = (vv.x - m[u]) * rs[u], h1 = (vv.y - m[u]) * rs[u], h2 = (vv.z - m[u]) * rs[u], h3 = (vv.w - m[u]) * rs[u];
                const float g0 = dd.x * g[k].x, g1 = dd.y * g[k].y, g2 = dd.z * g[k].z, g3 = dd.w * g[k].w;
                s1 += (g0 + g1) + (g2 + g3);
                s2 += (g0 * h0 + g1 * h1) + (g2 * h2 + g3 * h3);
                ca[k].x += dd.x * h0, ca[k].y += dd.y * h1, ca[k].z += dd.z * h2, ca[k].w += dd.w * h3;
                cb[k].x += dd.x, cb[k].y += dd.y, cb[k].z += dd.z, cb[k].w += dd.w;
            }
            s1 = wave_sum(s1);
            s2 = wave_sum(s2);
            if (lane == 0 && sums) reinterpret_cast<float2*>(sums)[r] = make_float2(s1, s2);
            if (WITH_DX) {
                // the pairs of all workers of this row, one worker per lane (at most 64 workers)
                float p1 = peer[u].x, p2 = peer[u].y;
                if (lane == dxa.my_part) p1 = s1, p2 = s2;
                const float S1 = wave_sum(p1) * dxa.weight, S2 = wave_sum(p2) * dxa.weight;
                T* dxr = static_cast<T*>(dxa.dx) + r * dxa.ld_dx;
#pragma unroll
                for (int k = 0; k < NV; ++k) {
                    const int c = lane + k * kWave;
                    if (c >= nv) continue;
                    const float4 dd = d[u][k], vv = v[u][k];
                    float4 o;
                    o.x = dx_value(dd.x, g[k].x, vv.x, m[u], rs[u], S1, S2);
                    o.y = dx_value(dd.y, g[k].y, vv.y, m[u], rs[u], S1, S2);
                    o.z = dx_value(dd.z, g[k].z, vv.z, m[u], rs[u], S1, S2);
                    o.w = dx_value(dd.w, g[k].w, vv.w, m[u], rs[u], S1, S2);
                    store_piece<ANY>(dxr + piece_column<ANY>(4 * c, n), o);
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c4 = (lane + k * kWave) * 4;
        if (ANY && c4 + 4 > n) {
            if (c4 >= n) continue;
            const int from = n - 4;
            const float a4[4] = {ca[k].x, ca[k].y, ca[k].z, ca[k].w}, b4[4] = {cb[k].x, cb[k].y, cb[k].z, cb[k].w};
#pragma unroll
            for (int e = 1; e < 4; ++e)
                if (from + e >= c4) fold[0][wave][from + e] = a4[e], fold[1][wave][from + e] = b4[e];
            continue;
        }
        *reinterpret_cast<float4*>(&fold[0][wave][c4]) = ca[k];
        *reinterpret_cast<float4*>(&fold[1][wave][c4]) = cb[k];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * static_cast<int>(cols); i += kFusedBlock) {
        const int which = i >= static_cast<int>(cols) ? 1 : 0, c = i - which * static_cast<int>(cols);
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < kFusedWaves; ++w) t += fold[which][w][c];
        partial[(static_cast<int64_t>(blockIdx.x) * 2 + which) * cols + c] = t;
    }
}

// Unaligned rows of fewer columns stay with the separate passes: measured with their ends fetched element by element,
// [30000, 801] bf16 107 -> 71 us in one pass (now 47), [8192, 1023] fp32 49 -> 27 (now 19), but [2048, 333] 10.4 -> 14 and
// [100000, 63] bf16 68 -> 92 (few lanes have a piece).
constexpr int64_t kAnyCols = 512;

template <typename T, bool WITH_DX, bool ANY>
void launch_partial_cols(const T* dy, const T* x, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x, const float* mean, const float* rstd,
                         const T* gamma, float* sums, int64_t splits, float* partial, const DxArgs& dxa, hipStream_t s) {
    const int64_t rows_per_split = (rows + splits - 1) / splits;
    auto go = [&](auto nv) {
        hipLaunchKernelGGL((ln_bwd_partial_cols<T, decltype(nv)::value, WITH_DX, ANY>), dim3(static_cast<uint32_t>(splits)), dim3(kFusedBlock), 0, s, dy,
                           x, rows, cols, ld_dy, ld_x, mean, rstd, gamma, sums, rows_per_split, partial, dxa);
    };
    if constexpr (!ANY) {
        if (cols <= kWave * 4) return go(std::integral_constant<int, 1>{});
        if (cols <= 2 * kWave * 4) return go(std::integral_constant<int, 2>{});
    }
    go(std::integral_constant<int, 4>{});
}

// Rows that do not fit a wavefront's registers, or are no multiple of four
// elements: the pass of ln_bwd_partial_cols with a workgroup per row.  Thread t
// keeps the pieces of four t + THREADS k, k < NV, of gamma and of the column
// sums in registers for all rows of its split; RU rows are loaded while the RU rows
// before them are summed, and the only barrier per RU rows is the exchange of the
// wavefronts' row sums (double-buffered in LDS).  Bound by HBM: dy and x are read
// once and dx written once.  [8192, 8192] bf16 measured, row sums + column sums + dx
// in separate passes 45 + 65 + 82 us, here together (see ddl_ln_bwd_whole_rows).  ANY:
// rows of any length, pitch and address, [8000, 8191] bf16 100 us one element a lane,
// here 81; [32000, 2045] 153 -> 102; the same in fp32 197 -> 141.
template <typename T, bool ANY>
struct Piece {
    struct __attribute__((packed, aligned((ANY ? 1 : 4) * sizeof(T)))) Raw {
        uint32_t word[sizeof(T)];   // four elements
    };
    static __device__ Raw fetch(const T* p) { return *reinterpret_cast<const Raw*>(p); }
    static __device__ void get(const Raw& r, float (&f)[4]) {
        struct __attribute__((aligned(4 * sizeof(T)))) Quad {
            uint32_t word[sizeof(T)];
        } w;
#pragma unroll
        for (int i = 0; i < static_cast<int>(sizeof(T)); ++i) w.word[i] = r.word[i];
        const float4 q = load4(reinterpret_cast<const T*>(&w));
        f[0] = q.x, f[1] = q.y, f[2] = q.z, f[3] = q.w;
    }
    static __device__ void put(T* p, const float (&f)[4]) { store_piece<ANY>(p, make_float4(f[0], f[1], f[2], f[3])); }
};

template <typename T, int THREADS, int NV, int RU, bool WITH_DX, bool ANY>
__global__ __launch_bounds__(THREADS) void ln_bwd_block_rows(const T* __restrict__ dy, const T* __restrict__ x, int64_t cols, int64_t ld_dy,
                                                             int64_t ld_x, const float* __restrict__ mean,
                                                             const float* __restrict__ rstd, const T* __restrict__ gamma,
                                                             float* __restrict__ sums, int rows_each, int rows_over, bool backwards,
                                                             float* __restrict__ partial, float weight, T* __restrict__ dx, int64_t ld_dx) {
#pragma clang fp contract(off)   // both instantiations round alike
    constexpr int V = 4;
    typedef Piece<T, ANY> P;
    typedef typename P::Raw Raw;
    constexpr int kWaves = THREADS / kWave;
    __shared__ float2 row_sums[2][RU][kWaves];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int n = static_cast<int>(cols), pieces = (n + V - 1) / V;
    auto column = [&](int c) { return piece_column<ANY>(V * c, n); };
    const int64_t splits = gridDim.x, own = rows_each + (static_cast<int>(blockIdx.x) < rows_over ? 1 : 0);   // rows of this split
    const int64_t first = backwards ? blockIdx.x + (own - 1) * splits : blockIdx.x, step = backwards ? -splits : splits;
    auto row_at = [&](int64_t i) { return first + i * step; };
    Raw g[NV];
    float ca[NV][V], cb[NV][V];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c = threadIdx.x + k * THREADS;
        if (gamma && c < pieces) g[k] = P::fetch(gamma + column(c));
#pragma unroll
        for (int e = 0; e < V; ++e) ca[k][e] = cb[k][e] = 0.f;
    }
    auto fetch = [&](int64_t r0, Raw (&d)[RU][NV], Raw (&v)[RU][NV], float (&m)[RU], float (&rs)[RU]) {
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const int64_t r = row_at(r0 + u < own ? r0 + u : own - 1);   // a row past the end repeats the last one and is not used
            m[u] = mean[r], rs[u] = rstd[r];
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int c = threadIdx.x + k * THREADS;
                if (c < pieces) {
                    d[u][k] = P::fetch(dy + r * ld_dy + column(c));
                    v[u][k] = P::fetch(x + r * ld_x + column(c));
                }
            }
        }
    };
    auto gain = [&](int k, float (&f)[V]) {
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = 1.f;
        if (gamma) P::get(g[k], f);
    };
    Raw d[RU][NV], v[RU][NV];
    float m[RU], rs[RU];
    if (own > 0) fetch(0, d, v, m, rs);
    int parity = 0;
    // Left in the middle, where `more` is false: with that as a condition of its own besides the loop's, the compiler sees a way round
    // on which the next rows' loads have not been waited for, and waits for each of them in front of the next.
    for (int64_t r0 = 0; own > 0; r0 += RU, parity ^= 1) {
        Raw d_next[RU][NV], v_next[RU][NV];
        float m_next[RU], rs_next[RU];
        const bool more = r0 + RU < own;
        if (more) fetch(r0 + RU, d_next, v_next, m_next, rs_next);
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            if (r0 + u >= own) break;   // the same in all threads
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                if (static_cast<int>(threadIdx.x) + k * THREADS >= pieces) continue;
                float dd[V], vv[V], gg[V];
                P::get(d[u][k], dd);
                P::get(v[u][k], vv);
                gain(k, gg);
                if (ANY) {
                    const int c = threadIdx.x + k * THREADS;
                    const float4 own = own_elements<ANY>(make_float4(dd[0], dd[1], dd[2], dd[3]), V * c - column(c));
                    dd[0] = own.x, dd[1] = own.y, dd[2] = own.z, dd[3] = own.w;
                }
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const float h = (vv[e] - m[u]) * rs[u], t = dd[e] * gg[e];
                    s1 += t;
                    s2 += t * h;
                    ca[k][e] += dd[e] * h;
                    cb[k][e] += dd[e];
                }
            }
            s1 = wave_sum(s1);
            s2 = wave_sum(s2);
            if (lane == 0) row_sums[parity][u][wave] = make_float2(s1, s2);
        }
        // Only LDS is exchanged: the loads of the next rows stay in flight.
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            if (r0 + u >= own) break;
            const int64_t r = row_at(r0 + u);
            const float2 p = lane < kWaves ? row_sums[parity][u][lane] : make_float2(0.f, 0.f);
            const float s1 = wave_sum(p.x), s2 = wave_sum(p.y);
            if (threadIdx.x == 0 && sums) reinterpret_cast<float2*>(sums)[r] = make_float2(s1, s2);
            if (WITH_DX) {
                const float S1 = s1 * weight, S2 = s2 * weight;
#pragma unroll
                for (int k = 0; k < NV; ++k) {
                    const int c = threadIdx.x + k * THREADS;
                    if (c >= pieces) continue;
                    if constexpr (NV * sizeof(T) == 16) {   // formed again: kept since the sums, h and t go to scratch memory
                        asm volatile("" : "+v"(m[u]));
#pragma unroll
                        for (int i = 0; i < static_cast<int>(sizeof(T)); ++i) asm volatile("" : "+v"(d[u][k].word[i]));
                    }
                    float dd[V], vv[V], gg[V], o[V];
                    P::get(d[u][k], dd);
                    P::get(v[u][k], vv);
                    gain(k, gg);
#pragma unroll
                    for (int e = 0; e < V; ++e) o[e] = dx_value(dd[e], gg[e], vv[e], m[u], rs[u], S1, S2);
                    P::put(dx + r * ld_dx + column(c), o);
                }
            }
        }
        if (!more) break;
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            m[u] = m_next[u], rs[u] = rs_next[u];
#pragma unroll
            for (int k = 0; k < NV; ++k) d[u][k] = d_next[u][k], v[u][k] = v_next[u][k];
        }
    }
    float* out = partial + static_cast<int64_t>(blockIdx.x) * 2 * cols;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c = threadIdx.x + k * THREADS;
        if (c >= pieces) continue;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const int at = column(c) + e;
            if (!ANY || at >= V * c) out[at] = ca[k][e], out[cols + at] = cb[k][e];
        }
    }
}

// The longest rows that ln_bwd_block_rows takes: what a workgroup's registers hold.
constexpr int64_t block_rows_cols(bool vec) { return vec ? 16384 : 8192; }

// Rows go to the workgroups in turn, so that those resident at one time work next to each other.  Where dy, x and dx are more
// than the Infinity Cache holds the last rows come first: dy has just been written, and x read, from the first row to the last.
// Training step of [8192, 8192] bf16, a run of rows to each workgroup -> so: 124.7 -> 123.3 us, with dy written right in front of it
// (and counted) 179.4 -> 171.0; [60000, 1100] 282.5 -> 271.7; fp32 [8192, 4096] 171.6 -> 170.1.  Smaller ones are better off
// in the usual order: [2048, 6000] 45.4 -> 44.9, but 46.2 with the last rows first.
// Rows of more than 8192 columns fill the registers.  With the two remarks in the kernel left out, runs of rows -> in turn: fp32 [1175, 8216]
// 31 -> 78 us, [2885, 11276] 82 -> 191, bf16 [2562, 11816] 45.6 -> 52.1; with them alike in bf16 and 1.02 to 1.09 times as fast in fp32.
constexpr int64_t kInfinityCache = 256ll << 20;

template <typename T, bool WITH_DX>
void launch_block_rows(bool vec, const T* dy, const T* x, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x, const float* mean,
                       const float* rstd, const T* gamma, float* sums, int64_t splits, float* partial, float weight, T* dx, int64_t ld_dx,
                       hipStream_t s) {
    const bool backwards = 3 * rows * cols * static_cast<int64_t>(sizeof(T)) > kInfinityCache;
    const int rows_each = static_cast<int>(rows / splits), rows_over = static_cast<int>(rows % splits);
    auto go_as = [&](auto threads, auto nv, auto ru, auto any) {
        constexpr int kThreads = decltype(threads)::value;
        hipLaunchKernelGGL((ln_bwd_block_rows<T, kThreads, decltype(nv)::value, decltype(ru)::value, WITH_DX, decltype(any)::value>),
                           dim3(static_cast<uint32_t>(splits)), dim3(kThreads), 0, s, dy, x, cols, ld_dy, ld_x, mean, rstd, gamma, sums,
                           rows_each, rows_over, backwards, partial, weight, dx, ld_dx);
    };
    auto go = [&](auto threads, auto nv, auto ru) {
        if (vec) go_as(threads, nv, ru, std::false_type{});
        else go_as(threads, nv, ru, std::true_type{});
    };
    const std::integral_constant<int, 1> c1{};
    const std::integral_constant<int, 2> c2{};
    const std::integral_constant<int, 4> c4{};
    const std::integral_constant<int, 512> c512{};
    const std::integral_constant<int, 1024> c1024{};
    if (cols <= 2048) go(c512, c1, c4);
    else if (cols <= 4096) go(c1024, c1, c4);
    else if (cols <= 8192) go(c1024, c2, c2);
    else go_as(c1024, c4, c1, std::false_type{});
}

// Can rows be read four elements at a time?  elem = bytes per element.
bool vectorizable(int elem, int64_t cols, std::initializer_list<int64_t> lds, std::initializer_list<const void*> ptrs) {
    if (cols % 4 != 0) return false;
    for (int64_t ld : lds)
        if (ld % 4 != 0) return false;
    for (const void* p : ptrs)
        if (p && !aligned_to(p, 4 * elem)) return false;
    return true;
}

int check_rows(const char* what, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x) {
    if (rows < 0 || cols < 1 || ld_dy < cols || ld_x < cols)
        return fail(DDL_E_ARG, "%s: rows=%lld cols=%lld ld_dy=%lld ld_x=%lld", what, (long long)rows, (long long)cols,
                    (long long)ld_dy, (long long)ld_x);
    if (rows > 0x7FFFFFFFll) return fail(DDL_E_UNSUPP, "%s: more than 2^31 rows", what);
    return 0;
}

int elem_bytes(int dtype) { return dtype == DDL_DT_F32 ? 4 : (dtype == DDL_DT_BF16 || dtype == DDL_DT_F16) ? 2 : 0; }

// Elements aligned to their own size, fp32 side arrays to 4 bytes, pairs to 8.
bool elems_aligned(int elem, std::initializer_list<const void*> ptrs) {
    for (const void* p : ptrs)
        if (p && !aligned_to(p, elem)) return false;
    return true;
}

// Row splits of the parameter gradients: as many as the workspace holds, at most
// 256 and at least `fewest` rows each.  0 when the workspace cannot hold one split.
int64_t param_splits(int64_t rows, int64_t cols, int64_t workspace_elems, int64_t fewest = 32) {
    int64_t splits = workspace_elems / (2 * cols);
    if (splits < 1) return 0;
    if (splits > 256) splits = 256;
    const int64_t by_rows = (rows + fewest - 1) / fewest;
    if (splits > by_rows) splits = by_rows > 0 ? by_rows : 1;
    return splits;
}

// Row splits of the sums over rows and columns together (ddl_ln_bwd_partial_params), for rows that ln_bwd_block_rows takes: one
// of 1024 threads fills a CU, so four rows each up to half the CUs; from there on eight, because the launch behind it reads the
// column sums of every split.  The times are at ddl_ln_bwd_partial_params.
int64_t block_row_splits(int64_t rows) {
    const int64_t four = (rows + 3) / 4, eight = (rows + 7) / 8;
    const int64_t splits = four < 128 ? four : eight < 128 ? 128 : eight < 256 ? eight : 256;
    return splits > 0 ? splits : 1;
}

bool by_block_rows(int64_t cols) { return cols > 4 * kWave * 4 && cols <= block_rows_cols(false); }

// With less room than that: splits for the two passes one after the other.
int64_t joint_splits(int64_t rows, int64_t cols, int64_t workspace_elems) {
    const int64_t splits = block_row_splits(rows);
    return by_block_rows(cols) && workspace_elems / (2 * cols) >= splits ? splits : param_splits(rows, cols, workspace_elems);
}

template <typename T>
const T* as(const void* p) { return static_cast<const T*>(p); }
template <typename T>
T* as(void* p) { return static_cast<T*>(p); }

}  // namespace
}  // namespace ddl

extern "C" int ddl_ln_bwd_partial(const void* dy, const void* x, int dtype, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                  const float* mean, const float* rstd, const void* gamma, float* sums, void* stream) {
    using namespace ddl;
    const int elem = elem_bytes(dtype);
    if (!elem) return fail(DDL_E_UNSUPP, "ln backward sums: dtype %d (f32, bf16, f16 only)", dtype);
    if (int rc = check_rows("ln backward sums", rows, cols, ld_dy, ld_x)) return rc;
    if (rows == 0) return 0;
    if (!dy || !x || !mean || !rstd || !sums) return fail(DDL_E_ARG, "ln backward sums: null pointer");
    if (!elems_aligned(elem, {dy, x, gamma}) || !aligned_to(mean, 4) || !aligned_to(rstd, 4) || !aligned_to(sums, 8))
        return fail(DDL_E_ALIGN, "ln backward sums: elements must be aligned to their size, mean and rstd to 4 bytes, the sums to 8");
    const uint32_t blocks = static_cast<uint32_t>((rows + kWavesPerBlock - 1) / kWavesPerBlock);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool vec = vectorizable(elem, cols, {ld_dy, ld_x}, {dy, x, gamma});
    with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        if (vec)
            hipLaunchKernelGGL((ln_bwd_partial<T, false>), dim3(blocks), dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), sums);
        else
            hipLaunchKernelGGL((ln_bwd_partial<T, true>), dim3(blocks), dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), sums);
    });
    return check_launch("ln_bwd_partial");
}

extern "C" int ddl_ln_bwd_input(const void* dy, const void* x, int dtype, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                const float* mean, const float* rstd, const void* gamma, const float* part_sums, int nparts,
                                float weight, void* dx, int64_t ld_dx, void* stream) {
    using namespace ddl;
    const int elem = elem_bytes(dtype);
    if (!elem) return fail(DDL_E_UNSUPP, "ln backward input: dtype %d (f32, bf16, f16 only)", dtype);
    if (int rc = check_rows("ln backward input", rows, cols, ld_dy, ld_x)) return rc;
    if (ld_dx < cols || nparts < 1) return fail(DDL_E_ARG, "ln backward input: ld_dx=%lld nparts=%d", (long long)ld_dx, nparts);
    if (rows == 0) return 0;
    if (!dy || !x || !mean || !rstd || !part_sums || !dx) return fail(DDL_E_ARG, "ln backward input: null pointer");
    if (!elems_aligned(elem, {dy, x, gamma, dx}) || !aligned_to(mean, 4) || !aligned_to(rstd, 4) || !aligned_to(part_sums, 8))
        return fail(DDL_E_ALIGN, "ln backward input: elements must be aligned to their size, mean and rstd to 4 bytes, the sums to 8");
    const uint32_t blocks = static_cast<uint32_t>((rows + kWavesPerBlock - 1) / kWavesPerBlock);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool vec = vectorizable(elem, cols, {ld_dy, ld_x, ld_dx}, {dy, x, gamma, dx});
    with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        if (vec)
            hipLaunchKernelGGL((ln_bwd_input<T, false>), dim3(blocks), dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd,
                               as<T>(gamma), part_sums, nparts, weight, as<T>(dx), ld_dx);
        else
            hipLaunchKernelGGL((ln_bwd_input<T, true>), dim3(blocks), dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd,
                               as<T>(gamma), part_sums, nparts, weight, as<T>(dx), ld_dx);
    });
    return check_launch("ln_bwd_input");
}

extern "C" int ddl_ln_bwd_params(const void* dy, const void* x, int dtype, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                 const float* mean, const float* rstd, void* dgamma, void* dbeta, float* workspace,
                                 int64_t workspace_elems, void* stream) {
    using namespace ddl;
    const int elem = elem_bytes(dtype);
    if (!elem) return fail(DDL_E_UNSUPP, "ln backward parameters: dtype %d (f32, bf16, f16 only)", dtype);
    if (int rc = check_rows("ln backward parameters", rows, cols, ld_dy, ld_x)) return rc;
    if (!dgamma && !dbeta) return 0;
    if (!workspace || (rows > 0 && (!dy || !x || !mean || !rstd))) return fail(DDL_E_ARG, "ln backward parameters: null pointer");
    if (!elems_aligned(elem, {dy, x, dgamma, dbeta}) || !aligned_to(mean, 4) || !aligned_to(rstd, 4) || !aligned_to(workspace, 4))
        return fail(DDL_E_ALIGN, "ln backward parameters: elements must be aligned to their size, fp32 arrays to 4 bytes");
    const int64_t splits = param_splits(rows, cols, workspace_elems);
    if (splits < 1) return fail(DDL_E_ARG, "ln backward parameters: workspace of %lld floats is smaller than 2 x %lld", (long long)workspace_elems, (long long)cols);
    const int64_t rows_per_split = rows > 0 ? (rows + splits - 1) / splits : 1;
    const int64_t strips = (cols + kStrip - 1) / kStrip;
    if (strips * splits > 0x7FFFFFFFll) return fail(DDL_E_UNSUPP, "ln backward parameters: too many workgroups");
    hipStream_t s = static_cast<hipStream_t>(stream);
    int rc = 0;
    with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        hipLaunchKernelGGL(ln_bwd_params_partial<T>, dim3(static_cast<uint32_t>(strips * splits)), dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows,
                           cols, ld_dy, ld_x, mean, rstd, rows_per_split, workspace, static_cast<int>(strips));
        rc = check_launch("ln_bwd_params_partial");
        if (rc) return;
        hipLaunchKernelGGL(ln_bwd_params_final<T>, dim3(static_cast<uint32_t>(strips)), dim3(kBlock), 0, s, workspace, cols,
                           static_cast<int>(splits), as<T>(dgamma), as<T>(dbeta));
        rc = check_launch("ln_bwd_params_final");
    });
    return rc;
}

extern "C" int64_t ddl_ln_bwd_partial_params_workspace(int64_t rows, int64_t cols) {
    using namespace ddl;
    if (rows < 0 || cols < 1) return 0;
    return 2 * cols * joint_splits(rows, cols, 512 * cols);
}

extern "C" int ddl_ln_bwd_partial_params(const void* dy, const void* x, int dtype, int64_t rows, int64_t cols, int64_t ld_dy,
                                         int64_t ld_x, const float* mean, const float* rstd, const void* gamma, float* sums,
                                         float* workspace, int64_t workspace_elems, void* stream) {
    using namespace ddl;
    const int elem = elem_bytes(dtype);
    if (!elem) return fail(DDL_E_UNSUPP, "ln backward sums: dtype %d (f32, bf16, f16 only)", dtype);
    if (int rc = check_rows("ln backward sums", rows, cols, ld_dy, ld_x)) return rc;
    if (!workspace) return fail(DDL_E_ARG, "ln backward sums: null workspace");
    const int64_t splits = joint_splits(rows, cols, workspace_elems);
    if (splits < 1) return fail(DDL_E_ARG, "ln backward sums: workspace of %lld floats is smaller than 2 x %lld", (long long)workspace_elems, (long long)cols);
    if (rows > 0 && (!dy || !x || !mean || !rstd || !sums)) return fail(DDL_E_ARG, "ln backward sums: null pointer");
    if (!elems_aligned(elem, {dy, x, gamma}) || !aligned_to(mean, 4) || !aligned_to(rstd, 4) || !aligned_to(sums, 8) || !aligned_to(workspace, 4))
        return fail(DDL_E_ALIGN, "ln backward sums: elements must be aligned to their size, fp32 arrays to 4 bytes, the sums to 8");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t rows_per_split = rows > 0 ? (rows + splits - 1) / splits : 1;
    const bool vec = vectorizable(elem, cols, {ld_dy, ld_x}, {dy, x, gamma});
    if (rows > 0 && cols <= 4 * kWave * 4 && (vec || cols > kAnyCols)) {
        with_ln_element(dtype, [&](auto* tag) {
            using T = std::remove_pointer_t<decltype(tag)>;
            if (vec)
                launch_partial_cols<T, false, false>(as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), sums, splits, workspace, DxArgs{}, s);
            else
                launch_partial_cols<T, false, true>(as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), sums, splits, workspace, DxArgs{}, s);
        });
        return check_launch("ln_bwd_partial_cols");
    }
    // One read of dy and x instead of two.  Event time with the dx launch, the two passes -> here: [5727, 4352] bf16 62.9 -> 49.3
    // us, fp32 103.9 -> 78.6; [2607, 2000] 20.9 -> 18.0; [1500, 5501] 40.5 -> 29.8; [1000, 4000] 25.2 -> 21.8; [512, 2176] 17.0 ->
    // 13.3; [256, 8192] 29.5 -> 22.7; fp32 rows of 1028 to 1531 columns are alike around 1000 of them (14.3 and 14.5).  In splits
    // of 32 rows [1024, 8192] took 58 us instead of 43.  Rows longer than those of by_block_rows: where every CU gets a split.
    if ((by_block_rows(cols) && splits == block_row_splits(rows)) || (splits == 256 && cols > 4 * kWave * 4 && cols <= block_rows_cols(vec))) {
        with_ln_element(dtype, [&](auto* tag) {
            using T = std::remove_pointer_t<decltype(tag)>;
            launch_block_rows<T, false>(vec, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), sums, splits, workspace, 0.f,
                                        static_cast<T*>(nullptr), 0, s);
        });
        return check_launch("ln_bwd_block_rows");
    }
    // everything else: the two passes separately, same results in the same places
    if (rows > 0) {
        if (int rc = ddl_ln_bwd_partial(dy, x, dtype, rows, cols, ld_dy, ld_x, mean, rstd, gamma, sums, stream)) return rc;
    }
    const int64_t strips = (cols + kStrip - 1) / kStrip;
    if (strips * splits > 0x7FFFFFFFll) return fail(DDL_E_UNSUPP, "ln backward sums: too many workgroups");
    with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        hipLaunchKernelGGL(ln_bwd_params_partial<T>, dim3(static_cast<uint32_t>(strips * splits)), dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows,
                           cols, ld_dy, ld_x, mean, rstd, rows_per_split, workspace, static_cast<int>(strips));
    });
    return check_launch("ln_bwd_params_partial");
}

extern "C" int ddl_ln_bwd_input_params(const void* dy, const void* x, int dtype, int64_t rows, int64_t cols, int64_t ld_dy,
                                       int64_t ld_x, const float* mean, const float* rstd, const void* gamma, const float* part_sums,
                                       int nparts, float weight, void* dx, int64_t ld_dx, const float* workspace,
                                       int64_t workspace_elems, void* dgamma, void* dbeta, void* stream) {
    using namespace ddl;
    const int elem = elem_bytes(dtype);
    if (!elem) return fail(DDL_E_UNSUPP, "ln backward input: dtype %d (f32, bf16, f16 only)", dtype);
    if (int rc = check_rows("ln backward input", rows, cols, ld_dy, ld_x)) return rc;
    if (ld_dx < cols || nparts < 1) return fail(DDL_E_ARG, "ln backward input: ld_dx=%lld nparts=%d", (long long)ld_dx, nparts);
    if (!workspace) return fail(DDL_E_ARG, "ln backward input: null workspace");
    const int64_t splits = joint_splits(rows, cols, workspace_elems);
    if (splits < 1) return fail(DDL_E_ARG, "ln backward input: workspace of %lld floats is smaller than 2 x %lld", (long long)workspace_elems, (long long)cols);
    if (rows > 0 && (!dy || !x || !mean || !rstd || !part_sums || !dx)) return fail(DDL_E_ARG, "ln backward input: null pointer");
    if (!elems_aligned(elem, {dy, x, gamma, dx, dgamma, dbeta}) || !aligned_to(mean, 4) || !aligned_to(rstd, 4) || !aligned_to(part_sums, 8) ||
        !aligned_to(workspace, 4))
        return fail(DDL_E_ALIGN, "ln backward input: elements must be aligned to their size, fp32 arrays to 4 bytes, the sums to 8");
    const int64_t input_blocks = (rows + kWavesPerBlock - 1) / kWavesPerBlock;
    const int64_t strips = (dgamma || dbeta) ? (cols + kStrip - 1) / kStrip : 0;
    if (input_blocks + strips == 0) return 0;
    if (input_blocks + strips > 0x7FFFFFFFll) return fail(DDL_E_UNSUPP, "ln backward input: too many workgroups");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<uint32_t>(input_blocks + strips));
    const bool vec = vectorizable(elem, cols, {ld_dy, ld_x, ld_dx}, {dy, x, gamma, dx});
    with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        if (vec)
            hipLaunchKernelGGL((ln_bwd_input_final<T, false>), grid, dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd,
                               as<T>(gamma), part_sums, nparts, weight, as<T>(dx), ld_dx, static_cast<uint32_t>(strips), workspace,
                               static_cast<int>(splits), as<T>(dgamma), as<T>(dbeta));
        else
            hipLaunchKernelGGL((ln_bwd_input_final<T, true>), grid, dim3(kBlock), 0, s, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd,
                               as<T>(gamma), part_sums, nparts, weight, as<T>(dx), ld_dx, static_cast<uint32_t>(strips), workspace,
                               static_cast<int>(splits), as<T>(dgamma), as<T>(dbeta));
    });
    return check_launch("ln_bwd_input_final");
}

extern "C" int ddl_ln_bwd_one_pass(const void* dy, const void* x, int dtype, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                   const float* mean, const float* rstd, const void* gamma, float* part_sums, int nparts, int my_part,
                                   float weight, void* dx, int64_t ld_dx, float* workspace, int64_t workspace_elems, void* dgamma,
                                   void* dbeta, void* stream) {
    using namespace ddl;
    const int elem = elem_bytes(dtype);
    if (!elem) return fail(DDL_E_UNSUPP, "ln backward (one pass): dtype %d (f32, bf16, f16 only)", dtype);
    if (int rc = check_rows("ln backward (one pass)", rows, cols, ld_dy, ld_x)) return rc;
    if (ld_dx < cols) return fail(DDL_E_ARG, "ln backward (one pass): ld_dx=%lld below cols=%lld", (long long)ld_dx, (long long)cols);
    if (nparts < 1 || nparts > kWave) return fail(DDL_E_UNSUPP, "ln backward (one pass): nparts=%d outside [1,%d]", nparts, kWave);
    if (my_part < 0 || my_part >= nparts) return fail(DDL_E_ARG, "ln backward (one pass): my_part=%d outside [0,%d)", my_part, nparts);
    if (nparts > 1 && !part_sums) return fail(DDL_E_ARG, "ln backward (one pass): the other workers' sums are missing");
    if (!workspace) return fail(DDL_E_ARG, "ln backward (one pass): null workspace");
    const int64_t splits = param_splits(rows, cols, workspace_elems);
    if (splits < 1) return fail(DDL_E_ARG, "ln backward (one pass): workspace of %lld floats is smaller than 2 x %lld", (long long)workspace_elems, (long long)cols);
    if (rows > 0 && (!dy || !x || !mean || !rstd || !dx)) return fail(DDL_E_ARG, "ln backward (one pass): null pointer");
    if (!elems_aligned(elem, {dy, x, gamma, dx, dgamma, dbeta}) || !aligned_to(mean, 4) || !aligned_to(rstd, 4) || !aligned_to(part_sums, 8) ||
        !aligned_to(workspace, 4))
        return fail(DDL_E_ALIGN, "ln backward (one pass): elements must be aligned to their size, fp32 arrays to 4 bytes, the sums to 8");
    if (cols > 4 * kWave * 4 || !vectorizable(elem, cols, {ld_dy, ld_x, ld_dx}, {dy, x, gamma, dx}))
        return fail(DDL_E_UNSUPP, "ln backward (one pass): rows of at most %d columns, columns and pitches multiples of 4, pointers aligned to 4 elements", 4 * kWave * 4);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t strips = (dgamma || dbeta) ? (cols + kStrip - 1) / kStrip : 0;
    if (rows > 0) {
        float* sums = part_sums ? part_sums + static_cast<int64_t>(my_part) * rows * 2 : nullptr;
        const DxArgs dxa{part_sums, nparts, my_part, weight, dx, ld_dx};
        with_ln_element(dtype, [&](auto* tag) {
            using T = std::remove_pointer_t<decltype(tag)>;
            launch_partial_cols<T, true, false>(as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), sums, splits, workspace, dxa, s);
        });
        if (int rc = check_launch("ln_bwd_partial_cols")) return rc;
    }
    if (strips == 0) return 0;
    with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        hipLaunchKernelGGL(ln_bwd_params_final<T>, dim3(static_cast<uint32_t>(strips)), dim3(kBlock), 0, s, workspace, cols,
                           static_cast<int>(rows > 0 ? splits : 0), as<T>(dgamma), as<T>(dbeta));
    });
    return check_launch("ln_bwd_params_final");
}

extern "C" int ddl_ln_bwd_whole_rows(const void* dy, const void* x, int dtype, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                     const float* mean, const float* rstd, const void* gamma, float weight, void* dx, int64_t ld_dx,
                                     float* workspace, int64_t workspace_elems, void* dgamma, void* dbeta, void* stream) {
    using namespace ddl;
    const int elem = elem_bytes(dtype);
    if (!elem) return fail(DDL_E_UNSUPP, "ln backward (whole rows): dtype %d (f32, bf16, f16 only)", dtype);
    if (int rc = check_rows("ln backward (whole rows)", rows, cols, ld_dy, ld_x)) return rc;
    if (ld_dx < cols) return fail(DDL_E_ARG, "ln backward (whole rows): ld_dx=%lld below cols=%lld", (long long)ld_dx, (long long)cols);
    const bool vec = vectorizable(elem, cols, {ld_dy, ld_x, ld_dx}, {dy, x, gamma, dx});
    if (cols <= kAnyCols || cols > block_rows_cols(vec))
        return fail(DDL_E_UNSUPP, "ln backward (whole rows): rows of %lld to %lld columns", (long long)kAnyCols + 1, (long long)block_rows_cols(vec));
    if (!workspace) return fail(DDL_E_ARG, "ln backward (whole rows): null workspace");
    // A workgroup per row: four rows per split already pay (a split's column sums are 8 bytes per column next to 4 rows x 3
    // tensors of elements).  A wavefront per row: eight rows at once.
    const bool by_wave = cols <= 4 * kWave * 4;
    const int64_t splits = param_splits(rows, cols, workspace_elems, by_wave ? 32 : 4);
    if (splits < 1) return fail(DDL_E_ARG, "ln backward (whole rows): workspace of %lld floats is smaller than 2 x %lld", (long long)workspace_elems, (long long)cols);
    if (rows > 0 && (!dy || !x || !mean || !rstd || !dx)) return fail(DDL_E_ARG, "ln backward (whole rows): null pointer");
    if (!elems_aligned(elem, {dy, x, gamma, dx, dgamma, dbeta}) || !aligned_to(mean, 4) || !aligned_to(rstd, 4) || !aligned_to(workspace, 4))
        return fail(DDL_E_ALIGN, "ln backward (whole rows): elements must be aligned to their size, fp32 arrays to 4 bytes");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (rows > 0) {
        with_ln_element(dtype, [&](auto* tag) {
            using T = std::remove_pointer_t<decltype(tag)>;
            if (by_wave)
                launch_partial_cols<T, true, true>(as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), nullptr, splits, workspace,
                                                   DxArgs{nullptr, 1, 0, weight, dx, ld_dx}, s);
            else
                launch_block_rows<T, true>(vec, as<T>(dy), as<T>(x), rows, cols, ld_dy, ld_x, mean, rstd, as<T>(gamma), nullptr, splits, workspace,
                                           weight, as<T>(dx), ld_dx, s);
        });
        if (int rc = check_launch("ln_bwd_block_rows")) return rc;
    }
    if (!dgamma && !dbeta) return 0;
    with_ln_element(dtype, [&](auto* tag) {
        using T = std::remove_pointer_t<decltype(tag)>;
        hipLaunchKernelGGL(ln_bwd_params_final<T>, dim3(static_cast<uint32_t>((cols + kStrip - 1) / kStrip)), dim3(kBlock), 0, s, workspace, cols,
                           static_cast<int>(rows > 0 ? splits : 0), as<T>(dgamma), as<T>(dbeta));
    });
    return check_launch("ln_bwd_params_final");
}

// The float32 forms.
extern "C" int ddl_ln_bwd_partial_f32(const float* dy, const float* x, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                      const float* mean, const float* rstd, const float* gamma, float* sums, void* stream) {
    return ddl_ln_bwd_partial(dy, x, DDL_DT_F32, rows, cols, ld_dy, ld_x, mean, rstd, gamma, sums, stream);
}
extern "C" int ddl_ln_bwd_input_f32(const float* dy, const float* x, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                    const float* mean, const float* rstd, const float* gamma, const float* part_sums,
                                    int nparts, float weight, float* dx, int64_t ld_dx, void* stream) {
    return ddl_ln_bwd_input(dy, x, DDL_DT_F32, rows, cols, ld_dy, ld_x, mean, rstd, gamma, part_sums, nparts, weight, dx, ld_dx, stream);
}
extern "C" int ddl_ln_bwd_params_f32(const float* dy, const float* x, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                     const float* mean, const float* rstd, float* dgamma, float* dbeta, float* workspace,
                                     int64_t workspace_elems, void* stream) {
    return ddl_ln_bwd_params(dy, x, DDL_DT_F32, rows, cols, ld_dy, ld_x, mean, rstd, dgamma, dbeta, workspace, workspace_elems, stream);
}
extern "C" int ddl_ln_bwd_partial_params_f32(const float* dy, const float* x, int64_t rows, int64_t cols, int64_t ld_dy,
                                             int64_t ld_x, const float* mean, const float* rstd, const float* gamma, float* sums,
                                             float* workspace, int64_t workspace_elems, void* stream) {
    return ddl_ln_bwd_partial_params(dy, x, DDL_DT_F32, rows, cols, ld_dy, ld_x, mean, rstd, gamma, sums, workspace, workspace_elems, stream);
}
extern "C" int ddl_ln_bwd_input_params_f32(const float* dy, const float* x, int64_t rows, int64_t cols, int64_t ld_dy, int64_t ld_x,
                                           const float* mean, const float* rstd, const float* gamma, const float* part_sums,
                                           int nparts, float weight, float* dx, int64_t ld_dx, const float* workspace,
                                           int64_t workspace_elems, float* dgamma, float* dbeta, void* stream) {
    return ddl_ln_bwd_input_params(dy, x, DDL_DT_F32, rows, cols, ld_dy, ld_x, mean, rstd, gamma, part_sums, nparts, weight, dx, ld_dx,
                                   workspace, workspace_elems, dgamma, dbeta, stream);
}
