// km_init.hpp -- initial centroids on the device (kmeans_init).
//
// Replaces kmeans_init's GPU kernels (cpp/oneapi/dal/algo/kmeans_init/backend/gpu/
// compute_kernels_impl.hpp:36-68 for dense, compute_kernel_distr_random_dense_dpc.cpp
// for random_dense) and adds plus_plus_dense, which the reference runs only on the
// host (its GPU kernel throws unimplemented; kmeans train without initial
// centroids calls DAAL's k-means++ on the CPU, train_kernel_lloyd_dense_dpc.cpp:44-74).
//
// k-means++ (D^2 sampling) here, in a fixed arithmetic order so that the oracle
// restates it bit for bit:
//   D2_r = min over chosen centroids of sum_f ((double)x_rf - (double)c_f)^2
//          (features in order, each sub/mul/add rounded separately);
//   chunk sums of OBJ_CHUNK rows (thread t of 256 sums rows t, t+256, ... in
//          order, then a tree of the 256 partials); group sums of INIT_GROUP
//          chunk sums each (in order); total = the group sums in order;
//   target = u * total with u from the counter RNG.  The walk descends with one
//          running sum: the first group whose running sum exceeds target (the
//          last group otherwise), then in it the first such chunk (its last
//          chunk otherwise), then in that chunk the first such block of
//          INIT_SUB rows (block sums in row order; its last block otherwise),
//          then in that block the first row with D2 > 0 whose running sum
//          exceeds target.  Rounding fallbacks: the block's last row with
//          D2 > 0, else the chunk's, else the chunk's first row.  If total is
//          0: row min(n - 1, floor(u * n)).
#pragma once

#include <cstdint>
#include <type_traits>

#include "km_common.hpp"

namespace km {

// chunk sums of v in the order of the file comment (one workgroup per chunk)
__global__ __launch_bounds__(256) void init_chunk_sums_kernel(const double* __restrict__ v, int64_t n,
                                                              double* __restrict__ chunk_sums) {
    __shared__ double part[256];
    const int t = threadIdx.x;
    const int64_t nchunks = (n + OBJ_CHUNK - 1) / OBJ_CHUNK;
    for (int64_t q = blockIdx.x; q < nchunks; q += gridDim.x) {
        const int64_t r0 = q * OBJ_CHUNK;
        const int rows = int(min<int64_t>(OBJ_CHUNK, n - r0));
        double p = 0.0;
        for (int r = t; r < rows; r += 256) p = p + v[r0 + r];
        __syncthreads();
        part[t] = p;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (t < s) part[t] = part[t] + part[t + s];
            __syncthreads();
        }
        if (t == 0) chunk_sums[q] = part[0];
    }
}

constexpr int INIT_GROUP = 64;  // chunk sums per group sum
constexpr int INIT_SUB = 16;    // rows per block of the last walk level

// The sampled row (one workgroup of 256): see the file comment.  Group sums and
// block sums are formed by all threads, each summing its own range in order (loads
// issued ahead); thread 0 does the short sequential walks.  gsum: INIT_GSUMS
// doubles of LDS.  Returns the row in every thread.
constexpr int INIT_GSUMS = 2048;  // group sums per LDS tile

__device__ __forceinline__ double init_group_sum(const double* __restrict__ chunk_sums, int64_t q0, int64_t q1) {
    double sg = 0.0;
    int64_t q = q0;
    for (; q + 16 <= q1; q += 16) {
        double w[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) w[u] = agent_load(chunk_sums + q + u);
#pragma unroll
        for (int u = 0; u < 16; ++u) sg = sg + w[u];
    }
    for (; q < q1; ++q) sg = sg + agent_load(chunk_sums + q);
    return sg;
}

// The walk over count sums in LDS: the first i with cum + v[i] > target (the last
// otherwise); cum then holds the sum before it.  One thread; sixteen values are
// loaded together, so the chain is the adds alone.
__device__ __forceinline__ int init_walk(const double* v, int count, double target, double& cum) {
    for (int i0 = 0; i0 < count; i0 += 16) {
        double w[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) w[u] = v[min(i0 + u, count - 1)];
        double c = cum;
        int sel = -1;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const double next = c + w[u];
            if (sel < 0) {
                if (next > target || i0 + u >= count - 1)
                    sel = i0 + u;
                else
                    c = next;
            }
        }
        cum = c;
        if (sel >= 0) return sel;
    }
    return count - 1;
}

__device__ __forceinline__ int64_t init_select(const double* __restrict__ D2, int64_t n,
                                               const double* __restrict__ chunk_sums, double u, double* gsum) {
    static_assert(OBJ_CHUNK / INIT_SUB <= 256, "one block sum per thread");
    __shared__ double bsum[OBJ_CHUNK / INIT_SUB];
    __shared__ double wrows[INIT_SUB];
    __shared__ double sh_total, sh_cum;
    __shared__ int64_t sh_sel;
    const int t = threadIdx.x;
    const int64_t nchunks = (n + OBJ_CHUNK - 1) / OBJ_CHUNK;
    const int64_t ngroups = (nchunks + INIT_GROUP - 1) / INIT_GROUP;
    auto tile_sums = [&](int64_t b, int m) {
        __syncthreads();
        for (int i = t; i < m; i += 256) {
            const int64_t q0 = (b + i) * INIT_GROUP;
            gsum[i] = init_group_sum(chunk_sums, q0, min<int64_t>(nchunks, q0 + INIT_GROUP));
        }
        __syncthreads();
    };
    int64_t qsel = 0;
    double cum = 0.0, target;
    if (nchunks == 1) {  // its group and chunk are the only ones
        const double total = agent_load(chunk_sums);
        if (!(total > 0.0)) {
            const double pos = u * double(n);
            return pos >= double(n - 1) ? n - 1 : int64_t(pos);
        }
        target = u * total;
    } else {
        // total = group sums in order
        double total = 0.0;
        for (int64_t b = 0; b < ngroups; b += INIT_GSUMS) {
            const int m = int(min<int64_t>(INIT_GSUMS, ngroups - b));
            tile_sums(b, m);
            if (t == 0)
                for (int i = 0; i < m; ++i) total = total + gsum[i];
        }
        if (t == 0) sh_total = total;
        __syncthreads();
        total = sh_total;
        if (!(total > 0.0)) {
            const double pos = u * double(n);
            return pos >= double(n - 1) ? n - 1 : int64_t(pos);
        }
        target = u * total;
        // the group
        int64_t gsel = -1;
        for (int64_t b = 0; b < ngroups; b += INIT_GSUMS) {
            const int m = int(min<int64_t>(INIT_GSUMS, ngroups - b));
            if (ngroups > INIT_GSUMS) tile_sums(b, m);  // one tile: still there
            if (t == 0 && gsel < 0) {
                const int i = init_walk(gsum, m, target, cum);
                if (b + m == ngroups || cum + gsum[i] > target)
                    gsel = b + i;
                else
                    cum = cum + gsum[i];  // the tile's last sum did not pass either
            }
        }
        // the chunk inside the group (its sums staged where the group sums were)
        if (t == 0) sh_sel = gsel;
        __syncthreads();
        gsel = sh_sel;
        const int64_t q0 = gsel * INIT_GROUP;
        const int nq = int(min<int64_t>(nchunks - q0, INIT_GROUP));
        if (t < nq) gsum[t] = agent_load(chunk_sums + q0 + t);
        __syncthreads();
        if (t == 0) {
            sh_sel = q0 + init_walk(gsum, nq, target, cum);
            sh_cum = cum;
        }
        __syncthreads();
        qsel = sh_sel;
        cum = sh_cum;
    }
    // block sums of the chunk: thread j sums rows INIT_SUB * j, ... in order
    const int64_t r0 = qsel * OBJ_CHUNK;
    const int rows = int(min<int64_t>(OBJ_CHUNK, n - r0));
    const int nb = (rows + INIT_SUB - 1) / INIT_SUB;
    if (t < nb) {
        double w[INIT_SUB], sb = 0.0;
#pragma unroll
        for (int r = 0; r < INIT_SUB; ++r) w[r] = t * INIT_SUB + r < rows ? D2[r0 + t * INIT_SUB + r] : 0.0;
#pragma unroll
        for (int r = 0; r < INIT_SUB; ++r)
            if (t * INIT_SUB + r < rows) sb = sb + w[r];
        bsum[t] = sb;
    }
    __syncthreads();
    if (t == 0) {
        sh_sel = init_walk(bsum, nb, target, cum);
        sh_cum = cum;
    }
    __syncthreads();
    const int jsel = int(sh_sel);
    const int rb = jsel * INIT_SUB, re = min(rows, rb + INIT_SUB);
    if (t < re - rb) wrows[t] = D2[r0 + rb + t];
    __syncthreads();
    if (t == 0) {
        int64_t idx = -1, last_pos = -1;
        double sr = sh_cum, w[INIT_SUB];
#pragma unroll
        for (int r = 0; r < INIT_SUB; ++r) w[r] = wrows[min(r, re - rb - 1)];
#pragma unroll
        for (int r = 0; r < INIT_SUB; ++r) {
            if (idx < 0 && rb + r < re) {
                if (w[r] > 0.0) last_pos = r0 + rb + r;
                sr = sr + w[r];
                if (w[r] > 0.0 && sr > target) idx = r0 + rb + r;
            }
        }
        if (idx < 0 && last_pos < 0) {
            for (int r = rows - 1; r >= 0; --r)
                if (D2[r0 + r] > 0.0) {
                    last_pos = r0 + r;
                    break;
                }
        }
        if (idx < 0) idx = last_pos >= 0 ? last_pos : r0;
        sh_sel = idx;
    }
    __syncthreads();
    return sh_sel;
}

__global__ __launch_bounds__(256) void init_select_kernel(const double* __restrict__ D2, int64_t n,
                                                         const double* __restrict__ chunk_sums, double u,
                                                         int64_t* __restrict__ chosen) {
    __shared__ double gsum[INIT_GSUMS];
    const int64_t row = init_select(D2, n, chunk_sums, u, gsum);
    if (threadIdx.x == 0) chosen[0] = row;
}

// ---------------------------------------------------------------------------
// One k-means++ step on dense rows.  init_step_kernel: D2 against the newest centroid
// (index t - 1, as doubles in cnew, zero-padded to whole pieces).  init_pick_kernel: the
// chunk sums, and by the last workgroup to finish the sampled row, which becomes
// centroid t (C and cnew).
//
// With thr, a row whose nearest centroid lies at least twice its distance away from
// the new one cannot get closer (triangle inequality; Elkan 2003 for k-means, Raff
// 2021 for this initialisation): thr_j = (||c_j - c_new|| / 2)^2, less 4e-6 of it for
// rounding, above D2 means that D2 stays, and the row is not read (12 bytes a row
// instead of d elements).  On clustered rows about half of the reads remain.
//
// A workgroup takes 256 U rows (U = 4, or 1 where that would leave the chip idle); each wave packs its open rows into a list and
// takes 64 at a time: PP lanes read one piece of PP x 16 bytes of a row, so for wide
// rows (PP = 8) every load is a full 128-byte line; the pieces pass through LDS
// (swizzled: 16-byte vector p of row r at p ^ (r % PP)) to the lane that owns the row,
// and the next piece's loads are in flight while a piece is summed.  Each D2 is
// summed in feature order; padding adds exact zeros.
// ---------------------------------------------------------------------------
// Rows up to which an item is 256 rows instead of 1024: a wave's four lists of 64 rows one after
// the other are the time of a step that has no work for the chip.  60 centroids on (n, d), items of
// 1024 and of 256 rows: (20000, 300) 4.66 and 2.12 ms, (1e5, 512) 7.32 and 3.63, (3e5, 128) 2.80 and
// 2.71, (5e5, 64) 2.45 and 2.56, (1e6, 64) 3.07 and 3.47, as fewer rows pack less well.
constexpr int64_t INIT_FEW_ROWS = 400000;

template <typename F>
struct init_step {
    const F* X;
    int64_t n;
    int d;
    int64_t t;          // centroids chosen so far (>= 1); the step adds centroid t
    const double* thr;  // t - 1 entries (null: every row is read)
    double* D2;
    int32_t* near;      // with thr: nearest chosen centroid of each row
    double* chunk_sums;
    double u;
    double* cnew;
    F* C;
    uint32_t* ticket;
};

template <typename F, int PP, int U>
__global__ __launch_bounds__(256, 4) void init_step_kernel(init_step<F> s) {
    constexpr int PART = 256 * U;           // rows per workgroup item
    constexpr int N = 16 / int(sizeof(F));  // elements per 16 bytes
    constexpr int FP = PP * N;              // features per piece
    constexpr int RL = 64 / PP;             // rows per load instruction
    typedef F V __attribute__((ext_vector_type(N)));
    typedef F VU __attribute__((ext_vector_type(N), aligned(sizeof(F))));  // rows of any width
    __shared__ __align__(16) V stage[4][64 * PP];
    __shared__ uint16_t list[4][PART / 4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int d = s.d;
    const int pieces = (d + FP - 1) / FP;
    const bool first = s.t == 1;
    const double* __restrict__ c = s.cnew;
    const int64_t nparts = (s.n + PART - 1) / PART;
    const uint64_t below = (uint64_t(1) << lane) - 1u;
    for (int64_t b = blockIdx.x; b < nparts; b += gridDim.x) {
        const int64_t r0 = b * PART;
        const int rows = int(min<int64_t>(PART, s.n - r0));
        int cnt = 0;
        {
            double v[U];
            int32_t nr[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int r = 256 * u + t;
                const bool look = s.thr && !first && r < rows;
                v[u] = look ? s.D2[r0 + r] : 0.0;
                nr[u] = look ? s.near[r0 + r] : -1;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int r = 256 * u + t;
                const bool open = r < rows && (nr[u] < 0 || !(s.thr[nr[u]] > v[u]));
                const uint64_t m = __ballot(open);
                if (open) list[wave][cnt + __popcll(m & below)] = uint16_t(r);
                cnt += __popcll(m);
            }
        }
        __builtin_amdgcn_wave_barrier();
        for (int g = 0; g < cnt; g += 64) {
            // lane loads: vector p = lane % PP of rows lane / PP + RL i
            const int p = lane % PP;
            const F* src[PP];
#pragma unroll
            for (int i = 0; i < PP; ++i) {
                const int e = min(cnt - 1, g + RL * i + lane / PP);
                src[i] = s.X + (r0 + list[wave][e]) * d + p * N;
            }
            // the lane's own row
            const int own = list[wave][min(cnt - 1, g + lane)];
            const double old = first ? 0.0 : s.D2[r0 + own];
            V v[PP];
            auto load = [&](int f0) {
                const int left = d - f0 - p * N;  // elements from this lane's vector to the row's end
#pragma unroll
                for (int i = 0; i < PP; ++i) {
                    V x{};
                    if (left >= N) {
                        x = *reinterpret_cast<const VU*>(src[i] + f0);
                    } else {
#pragma unroll
                        for (int e = 0; e < N - 1; ++e)
                            if (e < left) x[e] = src[i][f0 + e];
                    }
                    v[i] = x;
                }
            };
            load(0);
            double acc = 0.0;
            for (int pc = 0; pc < pieces; ++pc) {
#pragma unroll
                for (int i = 0; i < PP; ++i) {
                    const int r = RL * i + lane / PP;
                    stage[wave][r * PP + (p ^ (r % PP))] = v[i];
                }
                __builtin_amdgcn_wave_barrier();
                if (pc + 1 < pieces) load((pc + 1) * FP);
#pragma unroll
                for (int w = 0; w < PP; ++w) {
                    const V x = stage[wave][lane * PP + (w ^ (lane % PP))];
#pragma unroll
                    for (int e = 0; e < N; ++e) {
                        const double diff = double(x[e]) - c[pc * FP + w * N + e];
                        const double sq = diff * diff;
                        acc = acc + sq;
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
            if (g + lane < cnt && (first || acc < old || old != old)) {
                s.D2[r0 + own] = first ? acc : fmin(old, acc);
                if (s.thr) s.near[r0 + own] = int32_t(s.t - 1);
            }
        }
    }
}

template <typename F>
__global__ __launch_bounds__(256) void init_pick_kernel(init_step<F> s, int dp) {
    __shared__ double gsum[INIT_GSUMS];
    double* part = gsum;
    const int t = threadIdx.x;
    const int64_t nchunks = (s.n + OBJ_CHUNK - 1) / OBJ_CHUNK;
    for (int64_t q = blockIdx.x; q < nchunks; q += gridDim.x) {
        const int64_t r0 = q * OBJ_CHUNK;
        const int rows = int(min<int64_t>(OBJ_CHUNK, s.n - r0));
        constexpr int W = OBJ_CHUNK / 256;
        double v[W], sum = 0.0;
#pragma unroll
        for (int u = 0; u < W; ++u) v[u] = t + 256 * u < rows ? s.D2[r0 + t + 256 * u] : 0.0;
#pragma unroll
        for (int u = 0; u < W; ++u)
            if (t + 256 * u < rows) sum = sum + v[u];
        part[t] = sum;
        __syncthreads();
        for (int h = 128; h > 0; h >>= 1) {
            if (t < h) part[t] = part[t] + part[t + h];
            __syncthreads();
        }
        if (t == 0) agent_store(s.chunk_sums + q, part[0]);
        __syncthreads();
    }
    if (!last_workgroup(s.ticket)) return;
    const int64_t row = init_select(s.D2, s.n, s.chunk_sums, s.u, gsum);
    for (int f = t; f < dp; f += 256) {
        const F v = f < s.d ? s.X[row * s.d + f] : F(0);
        if (f < s.d) s.C[s.t * s.d + f] = v;
        s.cnew[f] = double(v);
    }
    if (t == 0) *s.ticket = 0u;
}

// thr_j of the step after centroid m was chosen (see init_step_kernel), j < m: one
// wave per centroid.  Distances near underflow or past the largest double skip nothing.
template <typename F>
__global__ __launch_bounds__(256) void init_pairs_kernel(const F* __restrict__ C, const double* __restrict__ cnew,
                                                         int64_t m, int d, double* __restrict__ thr) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = (int64_t(gridDim.x) * blockDim.x) >> 6;
    for (int64_t j = wave; j < m; j += nwaves) {
        double sq = 0.0;
        for (int f = lane; f < d; f += 64) {
            const double v = double(C[j * d + f]) - cnew[f];
            sq = fma(v, v, sq);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off);
        if (lane == 0) thr[j] = sq > 1e-280 && sq < 1e300 ? 0.25 * sq * (1.0 - 4e-6) : 0.0;
    }
}

// the first centroid: C[0] = X[row], also as doubles in cnew (dp entries, zeros past d)
template <typename F>
__global__ void init_first_kernel(const F* __restrict__ X, int d, int64_t row, F* __restrict__ C,
                                  double* __restrict__ cnew, int dp) {
    for (int f = threadIdx.x; f < dp; f += blockDim.x) {
        const F v = f < d ? X[row * d + f] : F(0);
        if (f < d) C[f] = v;
        cnew[f] = double(v);
    }
}

// C[i] = X[ids[i]] for i < k (random_dense); one workgroup per row
template <typename F>
__global__ void init_gather_rows_kernel(const F* __restrict__ X, int d, const int64_t* __restrict__ ids,
                                        int64_t k, F* __restrict__ C) {
    for (int64_t i = blockIdx.x; i < k; i += gridDim.x)
        for (int f = threadIdx.x; f < d; f += blockDim.x) C[i * d + f] = X[ids[i] * d + f];
}

// ---------------------------------------------------------------------------
// CSR rows.  The kernels below take rows whose column indices (minus `base`)
// increase strictly within each row; init_centroids_csr merges unsorted or repeated
// columns first.  A row then stands for its dense expansion: x_f = F(0) + v at
// a stored column f (the expansion adds each stored value to a zero), 0
// elsewhere.
// ---------------------------------------------------------------------------
constexpr int INIT_CSR_FT = 1024;  // centroid features staged per pass

// The D2 update on the dense expansion, without forming it: each thread walks
// its row's features in order (a missing feature contributes (0 - c_f)^2), so
// every sub, mul and add is the dense kernel's and D2 agrees bit for bit.
template <typename F>
__global__ __launch_bounds__(256) void init_d2_csr_kernel(const F* __restrict__ vals,
                                                          const int64_t* __restrict__ cols,
                                                          const int64_t* __restrict__ offs, int64_t base,
                                                          int64_t n, int d, const F* __restrict__ c,
                                                          double* __restrict__ D2, int first) {
    __shared__ double cs[INIT_CSR_FT];
    const int t = threadIdx.x;
    for (int64_t r0 = int64_t(blockIdx.x) * 256; r0 < n; r0 += int64_t(gridDim.x) * 256) {
        const int64_t r = r0 + t;
        const bool ok = r < n;
        int64_t p = ok ? offs[r] - base : 0;
        const int64_t e = ok ? offs[r + 1] - base : 0;
        int64_t nc = p < e ? cols[p] - base : INT64_MAX;  // next stored column
        double acc = 0.0;
        for (int f0 = 0; f0 < d; f0 += INIT_CSR_FT) {
            const int ft = min(INIT_CSR_FT, d - f0);
            __syncthreads();
            for (int q = t; q < ft; q += 256) cs[q] = double(c[f0 + q]);
            __syncthreads();
            if (ok) {
                for (int q = 0; q < ft; ++q) {
                    double xv = 0.0;
                    if (nc == int64_t(f0 + q)) {
                        xv = double(F(0) + vals[p]);
                        ++p;
                        nc = p < e ? cols[p] - base : INT64_MAX;
                    }
                    const double diff = xv - cs[q];
                    const double sq = diff * diff;
                    acc = acc + sq;
                }
            }
        }
        if (ok) D2[r] = first ? acc : fmin(D2[r], acc);
    }
}

// C[row_out + i] = dense expansion of row src_i for i < count: src_i = ids[i],
// or *chosen (count 1), or first + i; one workgroup per output row
template <typename F>
__global__ void init_expand_csr_rows_kernel(const F* __restrict__ vals, const int64_t* __restrict__ cols,
                                            const int64_t* __restrict__ offs, int64_t base, int d,
                                            const int64_t* __restrict__ ids, const int64_t* __restrict__ chosen,
                                            int64_t first, int64_t count, F* __restrict__ C, int64_t row_out) {
    for (int64_t i = blockIdx.x; i < count; i += gridDim.x) {
        const int64_t src = ids ? ids[i] : chosen ? chosen[0] : first + i;
        F* dst = C + (row_out + i) * int64_t(d);
        for (int f = threadIdx.x; f < d; f += blockDim.x) dst[f] = F(0);
        __syncthreads();  // zeros before the stored values (columns are distinct)
        const int64_t o0 = offs[src] - base, o1 = offs[src + 1] - base;
        for (int64_t p = o0 + threadIdx.x; p < o1; p += blockDim.x) dst[cols[p] - base] = F(0) + vals[p];
    }
}

}  // namespace km
