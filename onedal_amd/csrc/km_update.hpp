// km_update.hpp -- centroid update, objective and empty-cluster kernels.
//
// Replaces, on the oneDAL side:
//   count_clusters / count_empty_clusters   kernels_integral_dpc.cpp:45-149
//   partial_reduce_centroids                kernels_fp_impl.hpp:327-376
//   merge_reduce_centroids                  kernels_fp_impl.hpp:277-325
//   compute_objective_function              kernels_fp_impl.hpp:378-400
//   compute_squares (centroids)             kernels_fp_impl.hpp:402-414
//   find_candidates / fill_empty_clusters   empty_cluster_handling_dpc.cpp:26-150, 402-455
// The reference accumulates centroid sums in F with per-part copies walked by
// 128 subgroups; here rows are grouped by label (stable, ascending row index),
// each cluster's member list is cut into REDUCE_CHUNK chunks summed by one wave
// in double, and the chunk sums are merged in chunk order.  The order is fixed,
// so the result is identical run to run and identical to the oracle's
// restatement of it.
#pragma once

#include "km_bounds.hpp"
#include "km_common.hpp"

namespace km {

template <typename T>
__global__ void fill_kernel(T* __restrict__ p, int64_t count, T value) {
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < count;
         i += int64_t(gridDim.x) * blockDim.x)
        p[i] = value;
}

// copy rows into a zero-padded matrix with row stride ldx (for float4 row reads)
template <typename F>
__global__ void pad_rows_kernel(const F* __restrict__ X, int64_t n, int d, int64_t ldx,
                                F* __restrict__ out) {
    const int64_t total = n * ldx;
    for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < total;
         e += int64_t(gridDim.x) * blockDim.x) {
        const int64_t r = e / ldx;
        const int c = int(e - r * ldx);
        out[e] = c < d ? X[r * d + c] : F(0);
    }
}

// ---------------------------------------------------------------------------
// row norms: ||x_i|| rounded up to float (used only by the error bound)
// ---------------------------------------------------------------------------
template <typename F>
__global__ __launch_bounds__(256) void row_norm_kernel(const F* __restrict__ X, int64_t n, int d,
                                                       float* __restrict__ norm_up) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = (blockIdx.x * int64_t(blockDim.x) + threadIdx.x) >> 6;
    const int64_t nwaves = (int64_t(gridDim.x) * blockDim.x) >> 6;
    for (int64_t row = wave; row < n; row += nwaves) {
        double s = 0.0;
        for (int f = lane; f < d; f += 64) {
            const double v = double(X[row * d + f]);
            s = fma(v, v, s);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
        if (lane == 0) {
            const double r = sqrt(s) * (1.0 + 1e-12);
            float f = float(r);
            if (double(f) < r) f = __uint_as_float(__float_as_uint(f) + 1u);  // next float up (f >= 0)
            norm_up[row] = f;
        }
    }
}

// ---------------------------------------------------------------------------
// label histogram (count_clusters)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void count_kernel(const int32_t* __restrict__ labels, int64_t n,
                                                    int k, int32_t* __restrict__ counts,
                                                    int use_lds) {
    extern __shared__ int32_t hist[];
    if (use_lds) {
        for (int j = threadIdx.x; j < k; j += blockDim.x) hist[j] = 0;
        __syncthreads();
    }
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x) {
        const int j = labels[i];
        if (use_lds)
            atomicAdd(&hist[j], 1);
        else
            atomicAdd(&counts[j], 1);
    }
    if (use_lds) {
        __syncthreads();
        for (int j = threadIdx.x; j < k; j += blockDim.x)
            if (hist[j]) atomicAdd(&counts[j], hist[j]);
    }
}

// ---------------------------------------------------------------------------
// single-workgroup scan over clusters: member offsets, chunk offsets and the
// ascending list of empty clusters.  meta[0] = #empty, meta[1] = #chunks.  A
// cluster whose members did not change (changed[j] = 0) has no chunks: its sums,
// and so its centroid, are those of the previous iteration.  With gsum (the counting
// sort) the counts are first taken as its column sums over G groups.  The number
// of empty clusters also goes to host memory (report) with the number of rows that the
// pass assigned (*open; null: not told), followed by seq, so the host can leave out the
// refill's launches, or bounds that settle nothing, without waiting for the stream.
// ---------------------------------------------------------------------------
struct host_report {
    int32_t empties;
    int32_t open;
    uint32_t seq;
};

__device__ __forceinline__ void report_empties(host_report* report, int32_t empties, const int32_t* open, uint32_t seq) {
    if (!report) return;
    if (open) __hip_atomic_store(&report->open, *open, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&report->empties, empties, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&report->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// inclusive scans of three values over a workgroup of 1024 threads (sums: 16 x 3
// LDS words, rewritten by every call); returns this thread's inclusive values
__device__ __forceinline__ void scan3_1024(int32_t& a, int32_t& b, int32_t& c, int32_t (*sums)[16]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int32_t pa = __shfl_up(a, off), pb = __shfl_up(b, off), pc = __shfl_up(c, off);
        if (lane >= off) {
            a += pa;
            b += pb;
            c += pc;
        }
    }
    __syncthreads();  // the previous call's readers are done
    if (lane == 63) {
        sums[0][wave] = a;
        sums[1][wave] = b;
        sums[2][wave] = c;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) {
        a += sums[0][w];
        b += sums[1][w];
        c += sums[2][w];
    }
}

__global__ __launch_bounds__(1024) void scan_clusters_kernel(int32_t* __restrict__ counts,
                                                             const int32_t* __restrict__ gsum, int G,
                                                             int k,
                                                             int64_t* __restrict__ offsets,
                                                             int32_t* __restrict__ chunk_base,
                                                             int32_t* __restrict__ empty_list,
                                                             int32_t* __restrict__ meta,
                                                             const int32_t* __restrict__ changed,
                                                             host_report* report,
                                                             const int32_t* __restrict__ open, uint32_t seq) {
    __shared__ int32_t sums[3][16];
    __shared__ int32_t last[3];
    const int t = threadIdx.x;
    int32_t c_off = 0, c_chk = 0, c_emp = 0;  // of the earlier blocks of 1024 clusters
    for (int base = 0; base < k; base += 1024) {
        const int j = base + t;
        int32_t c = 0;
        if (j < k) {
            if (gsum) {
#pragma unroll 16
                for (int g = 0; g < G; ++g) c += gsum[int64_t(g) * k + j];
                counts[j] = c;
            } else {
                c = counts[j];
            }
        }
        const int32_t nchk = j < k && changed[j] ? (c + REDUCE_CHUNK - 1) / REDUCE_CHUNK : 0;
        int32_t so = c, sc = nchk, se = (j < k && c == 0) ? 1 : 0;  // the row count is below 2^31
        scan3_1024(so, sc, se, sums);
        if (j < k) {
            offsets[j] = int64_t(c_off) + so - c;
            chunk_base[j] = c_chk + sc - nchk;
            if (c == 0) empty_list[c_emp + se - 1] = j;
        }
        if (t == 1023) {
            last[0] = so;
            last[1] = sc;
            last[2] = se;
        }
        __syncthreads();
        c_off += last[0];
        c_chk += last[1];
        c_emp += last[2];
    }
    if (t == 0) {
        offsets[k] = c_off;
        chunk_base[k] = c_chk;
        meta[0] = c_emp;
        meta[1] = c_chk;
        report_empties(report, c_emp, open, seq);
    }
}

// ---------------------------------------------------------------------------
// Chunk sums.  One wave per chunk of REDUCE_CHUNK members of one cluster.
// G = reduce_groups(d) interleaved partial sums (member m of the chunk goes to
// partial m % G); lanes g*d + f (d <= 32) or f, f+64, ... (d > 32) own columns.
// CPL = columns per lane (d > 32 only).
// ---------------------------------------------------------------------------
template <typename F, int CPL>
__global__ __launch_bounds__(256) void reduce_chunks_kernel(
    const F* __restrict__ X, int d, int k, const int32_t* __restrict__ perm,
    const int64_t* __restrict__ offsets, const int32_t* __restrict__ chunk_base,
    const int32_t* __restrict__ meta, double* __restrict__ part) {
    const int lane = threadIdx.x & 63;
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int nwaves = (gridDim.x * blockDim.x) >> 6;
    const int total = meta[1];
    const int G = reduce_groups(d);
    const bool small = d <= 32;
    const int g = small ? lane / d : 0;
    const int f0 = small ? lane % d : lane;
    const bool active = small ? (g < G) : true;
    for (int q = wave; q < total; q += nwaves) {
        // cluster owning chunk q: last j with chunk_base[j] <= q
        int lo = 0, hi = k;  // chunk_base[k] = total > q
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (chunk_base[mid] <= q) lo = mid; else hi = mid;
        }
        const int j = lo;
        const int64_t m_begin = offsets[j] + int64_t(q - chunk_base[j]) * REDUCE_CHUNK;
        const int64_t m_end = min(m_begin + REDUCE_CHUNK, offsets[j + 1]);
        double acc[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[c] = 0.0;
        if (small) {
            int64_t m = m_begin;
            // eight steps of G members: ids and values loaded first, added in order
            for (; m + 8 * G <= m_end; m += 8 * G) {
                if (active) {
                    int64_t r[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) r[u] = perm[m + u * G + g];
                    double v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = double(X[r[u] * d + f0]);
#pragma unroll
                    for (int u = 0; u < 8; ++u) acc[0] = acc[0] + v[u];
                }
            }
            for (; m < m_end; m += G) {
                const int64_t mm = m + g;
                if (active && mm < m_end) {
                    const int64_t row = perm[mm];
                    acc[0] = acc[0] + double(X[row * d + f0]);
                }
            }
            // partial g -> group 0, added in g order
            double tot = acc[0];
            for (int gg = 1; gg < G; ++gg) {
                const double o = __shfl(acc[0], gg * d + f0);
                tot = tot + o;
            }
            if (g == 0 && f0 < d) part[int64_t(q) * d + f0] = tot;
        } else {
            int64_t m = m_begin;
            for (; m + 8 <= m_end; m += 8) {
                int64_t r[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) r[u] = perm[m + u];
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    const int f = f0 + 64 * c;
                    if (f < d) {
                        double v[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) v[u] = double(X[r[u] * d + f]);
#pragma unroll
                        for (int u = 0; u < 8; ++u) acc[c] = acc[c] + v[u];
                    }
                }
            }
            for (; m < m_end; ++m) {
                const int64_t r0 = perm[m];
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    const int f = f0 + 64 * c;
                    if (f < d) acc[c] = acc[c] + double(X[r0 * d + f]);
                }
            }
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const int f = f0 + 64 * c;
                if (f < d) part[int64_t(q) * d + f] = acc[c];
            }
        }
    }
}

// Same chunk sums for 32 < d <= 512 with d % 4 == 0 and 16-byte aligned rows:
// a sub-wave of lpc lanes (a power of two, lpc * 4 * V >= d) per chunk, lane l
// owning the 4-vectors l, l + lpc, ..., V of them, so a member's row is read with
// 16-byte loads (eight members' loads in flight).  Each feature is still summed
// over the chunk's members in order, so the partials equal reduce_chunks_kernel's.
template <typename F, int V>
__global__ __launch_bounds__(256) void reduce_chunks_vec_kernel(
    const F* __restrict__ X, int d, int k, const int32_t* __restrict__ perm,
    const int64_t* __restrict__ offsets, const int32_t* __restrict__ chunk_base,
    const int32_t* __restrict__ meta, double* __restrict__ part, int lpc) {
    typedef F F4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63;
    const int sub = lane / lpc, sl = lane - sub * lpc;
    const int subs = 64 / lpc;
    const int64_t gsub = int64_t((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * subs + sub;
    const int64_t nsub = int64_t((gridDim.x * blockDim.x) >> 6) * subs;
    const int total = meta[1];
    const int d4 = d / 4;
    for (int64_t q = gsub; q < total; q += nsub) {
        // cluster owning chunk q: last j with chunk_base[j] <= q
        int lo = 0, hi = k;  // chunk_base[k] = total > q
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (chunk_base[mid] <= q) lo = mid; else hi = mid;
        }
        const int j = lo;
        const int64_t m_begin = offsets[j] + int64_t(q - chunk_base[j]) * REDUCE_CHUNK;
        const int64_t m_end = min(m_begin + REDUCE_CHUNK, offsets[j + 1]);
        double acc[V][4];
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[v][e] = 0.0;
        int64_t m = m_begin;
        // member ids one batch ahead of the row loads (the row loads of a batch
        // then wait on one memory latency, not two)
        int32_t r[8];
        if (m + 8 <= m_end) {
#pragma unroll
            for (int u = 0; u < 8; ++u) r[u] = perm[m + u];
        }
        for (; m + 8 <= m_end; m += 8) {
            int32_t rn[8];
            const bool more = m + 16 <= m_end;
#pragma unroll
            for (int u = 0; u < 8; ++u) rn[u] = more ? perm[m + 8 + u] : 0;
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int c4 = sl + lpc * v;
                if (c4 < d4) {
                    F4 xv[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        xv[u] = *reinterpret_cast<const F4*>(X + int64_t(r[u]) * d + 4 * c4);
#pragma unroll
                    for (int u = 0; u < 8; ++u)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[v][e] = acc[v][e] + double(xv[u][e]);
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) r[u] = rn[u];
        }
        // the rest (fewer than eight): loads together, the valid ones added
        if (m < m_end) {
#pragma unroll
            for (int u = 0; u < 8; ++u) r[u] = perm[m + u < m_end ? m + u : m_begin];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int c4 = sl + lpc * v;
                if (c4 < d4) {
                    F4 xv[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        xv[u] = *reinterpret_cast<const F4*>(X + int64_t(r[u]) * d + 4 * c4);
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (m + u < m_end) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[v][e] = acc[v][e] + double(xv[u][e]);
                        }
                }
            }
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int c4 = sl + lpc * v;
            if (c4 < d4) {
                double* o = part + int64_t(q) * d + 4 * c4;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = acc[v][e];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// objective: d64 per row against its label's centroid (row_d64_kernel), then, in a
// fixed order: rows in chunks of OBJ_CHUNK; thread t of a chunk sums rows t, t+256,
// t+512, ... in order; the 256 partials are combined by the tree p[t] += p[t+s],
// s = 128..1; chunk sums are added in chunk order.
// ---------------------------------------------------------------------------
// d64 of every row: a wave takes 64 rows, a piece of PP 16-byte vectors at a time (PP = 8,
// less for rows of fewer vectors: at d = 2 seven of eight lanes would idle, n=1e6 28 us,
// 6.6 with PP = 1).
// PP lanes read a row's piece and their label's centroid's (so every load is whole
// lines: a lane reading its own row asks for a line per lane and load), form the squares
// and pass them through LDS (16-byte chunk q of row r at q ^ (r % chunks)) to the lane
// that owns the row, which adds them in feature order while the next piece's loads are in
// flight; past the last feature the squares are exact zeros.  Any width and alignment.
// Bound by HBM: n=2e7, d=128 3.25 -> 2.12 ms (4.8 TB/s), n=1e6, d=33 109 -> 44 us, n=3e5,
// d=50 in double 34 -> 29 us.
constexpr int D64_ROWS = 256;
template <typename F, int PP>
__global__ __launch_bounds__(256, 2) void row_d64_kernel(const F* __restrict__ X, int64_t n, int d,
                                                         const F* __restrict__ C,
                                                         const int32_t* __restrict__ labels,
                                                         double* __restrict__ d64) {
    constexpr int N = 16 / int(sizeof(F));  // elements per 16 bytes
    constexpr int FP = PP * N;              // features of a piece
    constexpr int RL = 64 / PP;             // rows per load instruction
    constexpr int CH = FP / 2;              // 16-byte chunks of a row's squares
    typedef F V __attribute__((ext_vector_type(N)));
    typedef F VU __attribute__((ext_vector_type(N), aligned(sizeof(F))));  // rows of any width
    typedef double D2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) D2 sq[4][64 * CH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = lane % PP;
    const int pieces = (d + FP - 1) / FP;
    for (int64_t w0 = int64_t(blockIdx.x) * D64_ROWS + 64 * wave; w0 < n; w0 += int64_t(gridDim.x) * D64_ROWS) {
        const int rows = int(min<int64_t>(64, n - w0));
        const int lab = labels[w0 + min(lane, rows - 1)];
        const F *xs[PP], *cs[PP];  // this lane's vector of rows lane / PP + RL i
#pragma unroll
        for (int i = 0; i < PP; ++i) {
            const int e = min(rows - 1, RL * i + lane / PP);
            xs[i] = X + (w0 + e) * d + p * N;
            cs[i] = C + int64_t(__shfl(lab, e)) * d + p * N;
        }
        V xv[PP], cv[PP];
        auto load = [&](int f0) {
            const int left = d - f0 - p * N;  // elements from this lane's vector to the row's end
#pragma unroll
            for (int i = 0; i < PP; ++i) {
                V x{}, c{};
                if (left >= N) {
                    x = *reinterpret_cast<const VU*>(xs[i] + f0);
                    c = *reinterpret_cast<const VU*>(cs[i] + f0);
                } else {
#pragma unroll
                    for (int e = 0; e < N - 1; ++e)
                        if (e < left) {
                            x[e] = xs[i][f0 + e];
                            c[e] = cs[i][f0 + e];
                        }
                }
                xv[i] = x;
                cv[i] = c;
            }
        };
        load(0);
        double acc = 0.0;
        for (int pc = 0; pc < pieces; ++pc) {
#pragma unroll
            for (int i = 0; i < PP; ++i) {
                const int r = RL * i + lane / PP;
#pragma unroll
                for (int u = 0; u < N / 2; ++u) {
                    const double da = double(xv[i][2 * u]) - double(cv[i][2 * u]);
                    const double db = double(xv[i][2 * u + 1]) - double(cv[i][2 * u + 1]);
                    sq[wave][r * CH + ((p * (N / 2) + u) ^ (r & (CH - 1)))] = D2{da * da, db * db};
                }
            }
            __builtin_amdgcn_wave_barrier();
            if (pc + 1 < pieces) load((pc + 1) * FP);
#pragma unroll
            for (int q = 0; q < CH; ++q) {
                const D2 v = sq[wave][lane * CH + (q ^ (lane & (CH - 1)))];
                acc = acc + v[0];
                acc = acc + v[1];
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (lane < rows) d64[w0 + lane] = acc;
    }
}

// Chunk sums of d64 and, by the last workgroup to finish (a ticket that it resets), the
// objective: the chunk sums added one at a time in chunk order onto `start` (null:
// 0).  The sum is bound by its chain of dependent adds, so the chunk sums are
// staged in LDS first.  The result also goes to host memory, when given: with the
// re-scored rows (counters, plus acc when not null), followed by seq.
struct objective_report {
    double value;
    unsigned long long refined[3];  // re-scored rows: candidate, full, collect
    uint32_t seq;
};
__device__ __forceinline__ void report_objective(objective_report* report, double value, const int32_t* counters,
                                                 const unsigned long long* acc, uint32_t seq) {
    __hip_atomic_store(&report->value, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    for (int q = 0; q < 3; ++q)
        __hip_atomic_store(&report->refined[q], (unsigned long long)counters[q] + (acc ? acc[q] : 0ull),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&report->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(256) void objective_sum_kernel(const double* __restrict__ d64, int64_t n,
                                                            double* __restrict__ chunk_sums,
                                                            const double* start, double* out,
                                                            objective_report* report, uint32_t seq,
                                                            const int32_t* __restrict__ counters,
                                                            const unsigned long long* __restrict__ acc,
                                                            uint32_t* __restrict__ ticket) {
    __shared__ double part[256];
    const int t = threadIdx.x;
    const int64_t nchunks = (n + OBJ_CHUNK - 1) / OBJ_CHUNK;
    for (int64_t q = blockIdx.x; q < nchunks; q += gridDim.x) {
        const int64_t r0 = q * OBJ_CHUNK;
        const int rows = int(min<int64_t>(OBJ_CHUNK, n - r0));
        constexpr int RPT = OBJ_CHUNK / 256;
        double v[RPT], p = 0.0;
#pragma unroll
        for (int u = 0; u < RPT; ++u) v[u] = t + 256 * u < rows ? d64[r0 + t + 256 * u] : 0.0;
#pragma unroll
        for (int u = 0; u < RPT; ++u)
            if (t + 256 * u < rows) p = p + v[u];
        part[t] = p;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (t < s) part[t] = part[t] + part[t + s];
            __syncthreads();
        }
        if (t == 0) agent_store(chunk_sums + q, part[0]);
        __syncthreads();
    }
    if (!last_workgroup(ticket)) return;
    double sum = start ? *start : 0.0;
    for (int64_t b = 0; b < nchunks; b += 256) {
        __syncthreads();
        if (b + t < nchunks) part[t] = agent_load(chunk_sums + b + t);
        __syncthreads();
        if (t == 0) {
            const int m = int(min<int64_t>(256, nchunks - b));
            int i = 0;
            for (; i + 16 <= m; i += 16) {
                double w[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) w[u] = part[i + u];
#pragma unroll
                for (int u = 0; u < 16; ++u) sum = sum + w[u];
            }
            for (; i < m; ++i) sum = sum + part[i];
        }
    }
    if (t == 0) {
        *out = sum;
        *ticket = 0u;
        if (report) report_objective(report, sum, counters, acc, seq);
    }
}

// the report alone (no objective asked for)
__global__ void refine_report_kernel(objective_report* report, const int32_t* counters,
                                     const unsigned long long* acc, uint32_t seq) {
    if (threadIdx.x == 0 && blockIdx.x == 0) report_objective(report, 0.0, counters, acc, seq);
}

// *out = v[0] + ... + v[count-1], added one at a time in order (one workgroup, the
// values staged in LDS)
__global__ __launch_bounds__(256) void sum_sequential_kernel(const double* __restrict__ v, int64_t count,
                                                             double* __restrict__ out) {
    __shared__ double part[256];
    double sum = 0.0;
    for (int64_t b = 0; b < count; b += 256) {
        const int m = int(min<int64_t>(256, count - b));
        __syncthreads();
        if (int(threadIdx.x) < m) part[threadIdx.x] = v[b + threadIdx.x];
        __syncthreads();
        if (threadIdx.x == 0) {
#pragma unroll 16
            for (int i = 0; i < m; ++i) sum = sum + part[i];
        }
    }
    if (threadIdx.x == 0) *out = sum;
}

// ---------------------------------------------------------------------------
// Empty clusters on the device, as a sequence of ordinary launches in the iterations
// that have any (m = meta[0] > 0; the host launches it when the scan reported some):
//   ec_hist_kernel x 8  radix select of the m-th largest d64, 8 bits a pass from
//                       the top (keys: the raw bits of the non-negative doubles,
//                       which order like the values); every workgroup derives
//                       the digits of the earlier passes from their histograms;
//   ec_count_kernel,    rows above the threshold (gt) and the first `remaining`
//   ec_collect_kernel   rows equal to it (eq), collected in row order (workgroup
//                       w owns a contiguous row range; block scans give in-order
//                       ranks);
//   ec_order_kernel     gt rows ordered by (d64 descending, row ascending), eq
//                       rows after them: pick e is the row with the e-th largest
//                       d64, ties to the lowest row;
//   ec_finish_kernel    pick e fills the e-th empty cluster (ascending index) of
//                       Cnext (dense rows; sparse rows are filled by
//                       csr_fill_empty_kernel from cand), and the objective (when
//                       given) drops by the picks' d64 in pick order.
// The d64 of every row against its label's centroid comes in (row_d64_kernel).
// ---------------------------------------------------------------------------
constexpr int EC_PASSES = 8;

// threshold state after `passes` radix passes: key prefix, its mask, and how
// many rows equal to the final key are still to be taken
__device__ __forceinline__ void ec_state(const unsigned int* __restrict__ hist, int passes, int m,
                                         unsigned long long& prefix, unsigned long long& mask,
                                         long long& rem) {
    prefix = 0ull;
    mask = 0ull;
    rem = m;
    for (int p = 0; p < passes; ++p) {
        const int shift = 56 - 8 * p;
        long long cum = 0;
        int digit = 0;
        for (int dg = 255; dg >= 0; --dg) {
            const long long c = hist[p * 256 + dg];
            if (cum + c >= rem) {
                digit = dg;
                rem -= cum;
                break;
            }
            cum += c;
        }
        prefix |= (unsigned long long)digit << shift;
        mask |= 0xFFull << shift;
    }
}

// the workgroup's copy of the state (thread 0 computes it)
__device__ __forceinline__ void ec_state_shared(const unsigned int* __restrict__ hist, int passes, int m,
                                                unsigned long long& prefix, unsigned long long& mask,
                                                long long& rem) {
    __shared__ unsigned long long s_prefix, s_mask;
    __shared__ long long s_rem;
    if (threadIdx.x == 0) ec_state(hist, passes, m, s_prefix, s_mask, s_rem);
    __syncthreads();
    prefix = s_prefix;
    mask = s_mask;
    rem = s_rem;
}

__device__ __forceinline__ unsigned long long ec_key(double v) {
    return (unsigned long long)__double_as_longlong(v);
}

__global__ __launch_bounds__(256) void ec_hist_kernel(const double* __restrict__ d64, int64_t n,
                                                      const int32_t* __restrict__ meta,
                                                      unsigned int* __restrict__ hist, int pass) {
    const int m = meta[0];
    if (m <= 0) return;
    __shared__ unsigned int h[256];
    unsigned long long prefix, mask;
    long long rem;
    ec_state_shared(hist, pass, m, prefix, mask, rem);
    const int shift = 56 - 8 * pass;
    h[threadIdx.x] = 0u;
    __syncthreads();
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const unsigned long long key = ec_key(d64[i]);
        if ((key & mask) == prefix) atomicAdd(&h[(key >> shift) & 0xFF], 1u);
    }
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&hist[pass * 256 + threadIdx.x], h[threadIdx.x]);
}

// workgroup w's contiguous row range
__device__ __forceinline__ void ec_range(int64_t n, int64_t& lo, int64_t& hi) {
    const int64_t span = (n + gridDim.x - 1) / gridDim.x;
    lo = min<int64_t>(n, int64_t(blockIdx.x) * span);
    hi = min<int64_t>(n, lo + span);
}

__global__ __launch_bounds__(256) void ec_count_kernel(const double* __restrict__ d64, int64_t n,
                                                       const int32_t* __restrict__ meta,
                                                       const unsigned int* __restrict__ hist,
                                                       int32_t* __restrict__ wcnt) {
    const int m = meta[0];
    if (m <= 0) return;
    __shared__ int32_t sa[256], sb[256];
    const int t = threadIdx.x;
    unsigned long long prefix, mask;
    long long rem;
    ec_state_shared(hist, EC_PASSES, m, prefix, mask, rem);
    int64_t lo, hi;
    ec_range(n, lo, hi);
    int cg_ = 0, ce = 0;
    for (int64_t i = lo + t; i < hi; i += 256) {
        const unsigned long long key = ec_key(d64[i]);
        cg_ += key > prefix;
        ce += key == prefix;
    }
    sa[t] = cg_;
    sb[t] = ce;
    __syncthreads();
    for (int s2 = 128; s2 > 0; s2 >>= 1) {
        if (t < s2) {
            sa[t] += sa[t + s2];
            sb[t] += sb[t + s2];
        }
        __syncthreads();
    }
    if (t == 0) {
        wcnt[2 * blockIdx.x] = sa[0];
        wcnt[2 * blockIdx.x + 1] = sb[0];
    }
}

__global__ __launch_bounds__(256) void ec_collect_kernel(const double* __restrict__ d64, int64_t n,
                                                         const int32_t* __restrict__ meta,
                                                         const unsigned int* __restrict__ hist,
                                                         const int32_t* __restrict__ wcnt,
                                                         int32_t* __restrict__ gt_list,
                                                         int32_t* __restrict__ eq_list) {
    const int m = meta[0];
    if (m <= 0) return;
    __shared__ int32_t sa[256], sb[256];
    const int t = threadIdx.x;
    unsigned long long prefix, mask;
    long long rem;
    ec_state_shared(hist, EC_PASSES, m, prefix, mask, rem);
    int64_t lo, hi;
    ec_range(n, lo, hi);
    // this workgroup's first gt and eq positions: the counts of the earlier ones
    long long bg = 0, be = 0;
    for (int w = t; w < int(blockIdx.x); w += 256) {
        bg += wcnt[2 * w];
        be += wcnt[2 * w + 1];
    }
    sa[t] = int(bg);
    sb[t] = int(be);
    __syncthreads();
    for (int s2 = 128; s2 > 0; s2 >>= 1) {
        if (t < s2) {
            sa[t] += sa[t + s2];
            sb[t] += sb[t + s2];
        }
        __syncthreads();
    }
    bg = sa[0];
    be = sb[0];
    __syncthreads();
    for (int64_t tile = lo; tile < hi; tile += 256) {
        const int64_t i = tile + t;
        bool fg = false, fe = false;
        if (i < hi) {
            const unsigned long long key = ec_key(d64[i]);
            fg = key > prefix;
            fe = key == prefix;
        }
        sa[t] = fg;
        sb[t] = fe;
        __syncthreads();
        for (int o = 1; o < 256; o <<= 1) {  // inclusive scans
            const int a = t >= o ? sa[t - o] : 0, b = t >= o ? sb[t - o] : 0;
            __syncthreads();
            sa[t] += a;
            sb[t] += b;
            __syncthreads();
        }
        if (fg) gt_list[bg + sa[t] - 1] = int32_t(i);
        if (fe && be + sb[t] - 1 < rem) eq_list[be + sb[t] - 1] = int32_t(i);
        bg += sa[255];
        be += sb[255];
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void ec_order_kernel(const double* __restrict__ d64,
                                                       const int32_t* __restrict__ meta,
                                                       const unsigned int* __restrict__ hist,
                                                       const int32_t* __restrict__ gt_list,
                                                       const int32_t* __restrict__ eq_list,
                                                       int32_t* __restrict__ cand, double* __restrict__ cand_d) {
    const int m = meta[0];
    if (m <= 0) return;
    unsigned long long prefix, mask;
    long long rem;
    ec_state_shared(hist, EC_PASSES, m, prefix, mask, rem);
    const long long ngt = m - rem;
    const int64_t gtid = int64_t(blockIdx.x) * 256 + threadIdx.x, gsize = int64_t(gridDim.x) * 256;
    for (long long i = gtid; i < ngt; i += gsize) {
        const int32_t ri = gt_list[i];
        const unsigned long long ki = ec_key(d64[ri]);
        long long rank = 0;
        for (long long j = 0; j < ngt; ++j) {
            const int32_t rj = gt_list[j];
            const unsigned long long kj = ec_key(d64[rj]);
            rank += (kj > ki) || (kj == ki && rj < ri);
        }
        cand[rank] = ri;
        cand_d[rank] = d64[ri];
    }
    for (long long e = gtid; e < rem; e += gsize) {
        cand[ngt + e] = eq_list[e];
        cand_d[ngt + e] = d64[eq_list[e]];
    }
}

template <typename F>
__global__ __launch_bounds__(256) void ec_finish_kernel(const F* __restrict__ X, int d,
                                                        const int32_t* __restrict__ meta,
                                                        const int32_t* __restrict__ empty_list,
                                                        const int32_t* __restrict__ cand,
                                                        const double* __restrict__ cand_d, F* __restrict__ Cnext,
                                                        double* __restrict__ obj) {
    const int m = meta[0];
    if (m <= 0) return;
    const int64_t gtid = int64_t(blockIdx.x) * 256 + threadIdx.x, gsize = int64_t(gridDim.x) * 256;
    if (X)
        for (int64_t e = gtid; e < int64_t(m) * d; e += gsize) {
            const int q = int(e / d), f = int(e - int64_t(q) * d);
            Cnext[int64_t(empty_list[q]) * d + f] = X[int64_t(cand[q]) * d + f];
        }
    if (gtid == 0 && obj) {
        double o = *obj;
        for (int e = 0; e < m; ++e) o = o - cand_d[e];
        *obj = o;
    }
}

}  // namespace km
