// km_bounds.hpp -- distance bounds that let a training pass skip settled rows.
//
// Hamerly's bounds (Hamerly 2010, "Making k-means even faster"; Elkan 2003): when
// a row is settled with label a, its distance to c_a is at most `up` and its
// distance to every other centroid at least `lo`.  Centroid j then moves by at
// most drift_j per iteration, so after some iterations the row's label is still
// a while  up + sum drift_a < lo - sum max_j drift_j.  One float per row is kept,
//     gap = lo (1 - g) - up (1 + g) + base_a            (rounded down)
// with base_a the running sum of (drift_a + max drift)(1 + g) (rounded up, in
// double) at the time the row was settled; the row stays settled while
//     gap > base_a + BOUND_SLACK.
// g covers the rounding of the exact-form distances D (their relative error is
// at most gamma_{d+2}), so a settled row's exact-form argmin is a, uniquely: the
// labels are those of a full pass, bit for bit.  BOUND_SLACK keeps the compared
// distances away from underflow, BOUND_MAX from overflow (such rows are always
// assigned again).  Any NaN makes the comparison false: the row is assigned again.
//
// What it is for: from the fourth iteration on, clustered rows move little and
// most labels are certain.  On the precision workload's mixture (n=2e7, d=128,
// k=1024, 20 iterations) 29% of the row assignments remain, on the FP32 one
// (n=1e7, d=64, k=256) 28%; where no row can be skipped a pass costs 8 bytes a
// row more (label and gap).
#pragma once

#include "km_common.hpp"

namespace km {

constexpr double BOUND_SLACK = 1e-15;
constexpr double BOUND_MAX = 1e18;

// rows of one assignment pass (null rows: all n) and where their bounds go
// (null gap: none kept)
struct row_select {
    const int32_t* rows;
    const int32_t* count;
    float* gap;
    const double* base;
    double gam;  // g above, with room for the float roundings of bound_gap
};

// the number of rows of the pass, and entry e's row
__device__ __forceinline__ int64_t select_rows(const row_select& s, int64_t n) {
    return s.rows ? int64_t(*s.count) : n;
}
__device__ __forceinline__ int64_t select_row(const row_select& s, int64_t e) {
    return s.rows ? int64_t(s.rows[e]) : e;
}

// the largest float at most v to within two roundings
__device__ __forceinline__ float float_below(double v) { return float(v - fabs(v) * 1.2e-7); }

// gap of a row settled with squared distances at most up2 (its centroid) and at
// least lo2 (every other one); the float roundings here are below 1e-6
__device__ __forceinline__ float bound_gap(double up2, double lo2, double gam, double base) {
    const float u = sqrtf(float(fmax(up2, 0.0)));
    const float l = sqrtf(float(fmax(lo2, 0.0)));
    if (!(double(u) < BOUND_MAX)) return -__builtin_inff();
    const double g = double(l) * (1.0 - gam) - double(u) * (1.0 + gam) + base;
    return float_below(g);
}

// gap of a row re-scored exactly: exact-form distances D1 (its centroid) and D2 (the
// next one re-scored), and a lower bound lo2 of the squared distance to the others;
// |D - dist^2| <= g dist^2
__device__ __forceinline__ float bound_gap_exact(double D1, double D2, double lo2, double gam, double base) {
    return bound_gap(D1 * (1.0 + 2.0 * gam), fmin(D2 * (1.0 - 2.0 * gam), lo2), gam, base);
}

// The rows to assign again, as a dense list.  A workgroup takes runs of
// SELECT_ROWS rows: a lane holds four consecutive rows of each of its wave's groups
// of 256 (16-byte loads), positions inside the run come from four ballots, and one
// atomic reserves the run's part of the list; rows keep their order inside a run.
// 8 bytes read per row: bound by HBM.
constexpr int SELECT_ROWS = 4096;
__global__ __launch_bounds__(256) void bound_select_kernel(const int32_t* __restrict__ labels,
                                                           const float* __restrict__ gap,
                                                           const double* __restrict__ base, int64_t n,
                                                           int32_t* __restrict__ rows,
                                                           int32_t* __restrict__ count) {
    typedef int I4 __attribute__((ext_vector_type(4)));
    typedef float F4 __attribute__((ext_vector_type(4)));
    constexpr int U = SELECT_ROWS / 1024;
    __shared__ int wtot[4];
    __shared__ int first;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t below = (uint64_t(1) << lane) - 1u;
    const int64_t runs = (n + SELECT_ROWS - 1) / SELECT_ROWS;
    for (int64_t q = blockIdx.x; q < runs; q += gridDim.x) {
        const int64_t r0 = q * SELECT_ROWS + int64_t(wave) * (SELECT_ROWS / 4) + 4 * lane;
        I4 lab[U];
        F4 g[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t r = r0 + 256 * u;
            if (r + 4 <= n) {
                lab[u] = *reinterpret_cast<const I4*>(labels + r);
                g[u] = *reinterpret_cast<const F4*>(gap + r);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    lab[u][e] = r + e < n ? labels[r + e] : 0;
                    g[u][e] = r + e < n ? gap[r + e] : 0.f;
                }
            }
        }
        uint64_t open[U][4];
        int mine = 0;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool settled = double(g[u][e]) > base[lab[u][e]] + BOUND_SLACK;
                open[u][e] = __ballot(r0 + 256 * u + e < n && !settled);
                mine += __popcll(open[u][e]);
            }
        if (lane == 0) wtot[wave] = mine;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int t = wtot[0] + wtot[1] + wtot[2] + wtot[3];
            first = t ? atomicAdd(count, t) : 0;
        }
        __syncthreads();
        int at = first;
        for (int w = 0; w < wave; ++w) at += wtot[w];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int p = at;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                p += __popcll(open[u][e] & below);
                at += __popcll(open[u][e]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if ((open[u][e] >> lane) & 1u) rows[p++] = int32_t(r0 + 256 * u + e);
        }
        __syncthreads();  // wtot and first are rewritten by the next run
    }
}

}  // namespace km
