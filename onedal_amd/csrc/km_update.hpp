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
// of empty clusters also goes to host memory (report), followed by seq, so the
// host can leave out the refill's launches without waiting for the stream.
// ---------------------------------------------------------------------------
struct host_report {
    int32_t empties;
    uint32_t seq;
};

__device__ __forceinline__ void report_empties(host_report* report, int32_t empties, uint32_t seq) {
    if (!report) return;
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
                                                             host_report* report, uint32_t seq) {
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
        report_empties(report, c_emp, seq);
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
// d64 of one row, features in order: 16-byte loads, a 128-byte line of the row and of
// the centroid per step, when vec (whole 16-byte pieces, 16-byte aligned)
template <typename F>
__device__ __forceinline__ double row_d64(const F* __restrict__ x, const F* __restrict__ c, int d, bool vec) {
    typedef F V __attribute__((ext_vector_type(16 / int(sizeof(F)))));
    constexpr int N = 16 / int(sizeof(F));  // elements per 16 bytes
    double acc = 0.0;
    int f = 0;
    if (vec) {
        for (; f + 8 * N <= d; f += 8 * N) {
            V xv[8], cv[8];
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                xv[v] = *reinterpret_cast<const V*>(x + f + N * v);
                cv[v] = *reinterpret_cast<const V*>(c + f + N * v);
            }
#pragma unroll
            for (int v = 0; v < 8; ++v)
#pragma unroll
                for (int e = 0; e < N; ++e) {
                    const double diff = double(xv[v][e]) - double(cv[v][e]);
                    const double sq = diff * diff;
                    acc = acc + sq;
                }
        }
        for (; f < d; f += N) {
            const V xv = *reinterpret_cast<const V*>(x + f);
            const V cv = *reinterpret_cast<const V*>(c + f);
#pragma unroll
            for (int e = 0; e < N; ++e) {
                const double diff = double(xv[e]) - double(cv[e]);
                const double sq = diff * diff;
                acc = acc + sq;
            }
        }
    }
    for (; f < d; ++f) {
        const double diff = double(x[f]) - double(c[f]);
        const double sq = diff * diff;
        acc = acc + sq;
    }
    return acc;
}

// One row per thread, 256 rows per workgroup.  Rows that allow 16-byte reads are read
// directly.  The others (odd widths) are contiguous in memory as a block: the
// workgroup copies up to FT features of its 256 rows to LDS in consecutive
// elements and each thread then walks its own row there (row stride odd, so the
// lanes meet different banks), the centroid from the cache.
constexpr int D64_ROWS = 256;
template <typename F>
__global__ __launch_bounds__(256) void row_d64_kernel(const F* __restrict__ X, int64_t n, int d,
                                                      const F* __restrict__ C,
                                                      const int32_t* __restrict__ labels,
                                                      double* __restrict__ d64) {
    constexpr int FT = 96 / int(sizeof(F));  // staged features: 24 float, 12 double
    constexpr int ST = FT | 1;
    __shared__ F Xs[D64_ROWS * ST];
    const int t = threadIdx.x;
    constexpr int N = 16 / int(sizeof(F));
    const bool vec = (d % N) == 0 && (reinterpret_cast<uintptr_t>(X) % 16) == 0 &&
                     (reinterpret_cast<uintptr_t>(C) % 16) == 0;
    for (int64_t r0 = int64_t(blockIdx.x) * D64_ROWS; r0 < n; r0 += int64_t(gridDim.x) * D64_ROWS) {
        const int nr = int(min<int64_t>(D64_ROWS, n - r0));
        const F* c = C + int64_t(t < nr ? labels[r0 + t] : 0) * d;
        if (vec) {
            if (t < nr) d64[r0 + t] = row_d64<F>(X + (r0 + t) * d, c, d, true);
            continue;
        }
        double acc = 0.0;
        for (int f0 = 0; f0 < d; f0 += FT) {
            const int ft = min(FT, d - f0);
            __syncthreads();
            if (ft == d) {  // whole rows: one contiguous run
                for (int e = t; e < nr * d; e += 256) {
                    const int r = e / d;
                    Xs[r * ST + (e - r * d)] = X[r0 * d + e];
                }
            } else {
                for (int e = t; e < nr * FT; e += 256) {
                    const int r = e / FT, f = e - r * FT;
                    if (f < ft) Xs[r * ST + f] = X[(r0 + r) * d + f0 + f];
                }
            }
            __syncthreads();
            if (t < nr) {
                for (int f = 0; f < ft; ++f) {
                    const double diff = double(Xs[t * ST + f]) - double(c[f0 + f]);
                    const double sq = diff * diff;
                    acc = acc + sq;
                }
            }
        }
        if (t < nr) d64[r0 + t] = acc;
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
