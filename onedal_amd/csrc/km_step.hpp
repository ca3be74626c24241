// km_step.hpp -- the centroid step between two assignment passes, and the grouping of
// few rows.
//
// One launch merges the chunk sums into the new centroids (merge_reduce_centroids,
// kernels_fp_impl.hpp:277-325), prepares them for the next pass (norms, padded or
// BF16 copies, their maxima; compute_squares :402-414), takes how far they moved and
// advances the bounds (km_bounds.hpp).  These were five to seven launches of a few
// microseconds each, which set the time of small trainings: n=10000, d=20, k=10
// ran at 107 us an iteration for 30 launches.
#pragma once

#include "km_assign_bf16.hpp"
#include "km_assign_split.hpp"
#include "km_assign_wide.hpp"
#include "km_bounds.hpp"
#include "km_common.hpp"
#include "km_update.hpp"

namespace km {

constexpr int STEP_MAX_GRID = 256;

// feature f of the chunk sums q0 .. q1 - 1, added in chunk order (loads issued ahead)
__device__ __forceinline__ double merge_chunks(const double* __restrict__ part, int q0, int q1, int d, int f) {
    double sum = 0.0;
    int q = q0;
    for (; q + 16 <= q1; q += 16) {
        double w[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) w[u] = part[int64_t(q + u) * d + f];
#pragma unroll
        for (int u = 0; u < 16; ++u) sum = sum + w[u];
    }
    for (; q < q1; ++q) sum = sum + part[int64_t(q) * d + f];
    return sum;
}

// Wide rows (d > STEP_MERGE_D): the merge and the division in a launch of their own, a
// workgroup per centroid and 256 features, as the step's one workgroup per centroid
// would read all of a large cluster's chunk sums (d = 2000, a cluster with a third of
// n=1e6 rows: 480 us in the step, 63 us here; up to two slabs the extra launch costs more
// than it gives: 5 us).
constexpr int STEP_MERGE_D = 512;
template <typename F>
__global__ __launch_bounds__(256) void merge_centroids_kernel(const double* __restrict__ part,
                                                              const int32_t* __restrict__ counts,
                                                              const int32_t* __restrict__ chunk_base,
                                                              const int32_t* __restrict__ changed, int k, int d,
                                                              const F* __restrict__ cold, F* __restrict__ C) {
    const int slabs = (d + 255) / 256;
    for (int64_t e = blockIdx.x; e < int64_t(k) * slabs; e += gridDim.x) {
        const int j = int(e / slabs), f = int(e % slabs) * 256 + threadIdx.x;
        if (f >= d) continue;
        const int64_t o = int64_t(j) * d + f;
        const int32_t cnt = counts[j];
        C[o] = cnt == 0 || !changed[j] ? cold[o]
                                       : F(merge_chunks(part, chunk_base[j], chunk_base[j + 1], d, f) / double(cnt));
    }
}

// the bf16 pieces of v, `stride` apart
__device__ __forceinline__ void split_feature(float v, uint16_t* out, int stride) {
#pragma unroll
    for (int p = 0; p < SPLIT_PIECES; ++p) {
        const uint16_t b = f2bf(v);
        out[p * stride] = b;
        v -= bf2f(b);
    }
}

template <typename F>
struct centroid_step {
    // new centroids from the chunk sums (null part: C holds them already)
    const double* part;
    const int32_t* counts;
    const int32_t* chunk_base;
    F* C;
    const F* cold;  // previous centroids (null: a first pass, no bounds)
    int k, d, dpad;
    // for the assignment: ||c_j||^2, and a zero-padded copy (cpad) or bf16(-2 c) rows
    // (Cb, kp rows, those past k zero); null where the path does not read them
    F* cn;
    F* cpad;
    uint16_t* Cb;
    // or (Csp) rows of the three bf16 pieces of -2 c and (cnp) the pieces of ||c_j||^2 for the
    // norm step of assign_split_kernel, kp rows
    uint16_t* Csp;
    uint16_t* cnp;
    // or (Cw) the pieces chunk by chunk for assign_wide_kernel, kp rows, and their norms
    uint16_t* Cw;
    float* cnw;
    int kp;
    double* maxima;  // [0] max ||c||, with Cb or Csp: [1] max ||bf16(c)||, [2] max ||c - bf16(c)||
    // BF16: value shift and start values
    const unsigned long long* xmax_bits;
    bf16_consts kc;
    bf16_params* params;
    float* cnb;
    // bounds (cold not null)
    double* drift;
    double* base;
    double gam;
    int32_t* changed;
    int32_t* sel_count;
    // re-score counters: added into acc (when not null), then cleared
    int32_t* counters;
    unsigned long long* acc;
    // workspace of the launch: a ticket (0 between launches) and STEP_MAX_GRID x 4 maxima
    uint32_t* ticket;
    unsigned long long* wgmax;
};

// A workgroup takes every gridDim-th centroid: the chunk sums in chunk order and the
// division (an unchanged cluster keeps its bits, an empty one is left as it was for
// the ec_* kernels), then the first wave the norms (double sums over lanes).  The
// maxima are the bits of non-negative doubles (a NaN wins); one entry per workgroup,
// joined by the last workgroup to finish (a ticket that it resets), which advances
// base_j += (drift_j + max drift)(1 + g), rounded up, and clears the pass's counters.
template <typename F, bool BF16>
__global__ __launch_bounds__(256) void centroid_step_kernel(centroid_step<F> s) {
    extern __shared__ __align__(16) unsigned char step_raw[];
    F* row = reinterpret_cast<F*>(step_raw);  // [d]
    __shared__ unsigned long long red[4][4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int k = s.k, d = s.d, dpad = s.dpad;
    unsigned long long mx[4] = {0ull, 0ull, 0ull, 0ull};  // wave 0, lane 0
    for (int j = blockIdx.x; j < k; j += gridDim.x) {
        const int64_t o = int64_t(j) * d;
        if (s.part) {
            const int32_t cnt = s.counts[j];
            const bool keep = cnt == 0 || !s.changed[j];
            const int q0 = s.chunk_base[j], q1 = s.chunk_base[j + 1];
            for (int f = t; f < d; f += 256) {
                const F v = keep ? s.cold[o + f] : F(merge_chunks(s.part, q0, q1, d, f) / double(cnt));
                s.C[o + f] = v;
                row[f] = v;
            }
        } else {
            for (int f = t; f < d; f += 256) row[f] = s.C[o + f];
        }
        __syncthreads();
        if constexpr (BF16) {
            for (int f = t; f < dpad; f += 256)  // exact: -2 * bf16(c)
                s.Cb[int64_t(j) * dpad + f] = f < d ? f2bf(-2.0f * bf2f(f2bf(float(row[f])))) : uint16_t(0);
        } else if (s.Csp) {
            uint16_t* o3 = s.Csp + int64_t(j) * SPLIT_PIECES * dpad;
            for (int f = t; f < dpad; f += 256) split_feature(f < d ? -2.0f * float(row[f]) : 0.f, o3 + f, dpad);
        } else if (s.Cw) {
            for (int f = t; f < 32 * wide_chunks(d); f += 256) {
                uint16_t* o3 = s.Cw + (int64_t(f >> 5) * s.kp + j) * WIDE_ROW + (f & 31);
                split_feature(f < d ? -2.0f * float(row[f]) : 0.f, o3, 32);
            }
        } else if (s.cpad) {
            for (int f = t; f < dpad; f += 256) s.cpad[int64_t(j) * dpad + f] = f < d ? row[f] : F(0);
        }
        if (wave == 0) {
            double sq = 0.0, sh = 0.0, se = 0.0, sd = 0.0;
            for (int f = lane; f < d; f += 64) {
                const double v = double(row[f]);
                sq = fma(v, v, sq);
                if (BF16 || s.Csp) {
                    const double vh = double(bf2f(f2bf(float(row[f])))), ve = v - vh;
                    sh = fma(vh, vh, sh);
                    se = fma(ve, ve, se);
                }
                if (s.cold) {
                    const double m = v - double(s.cold[o + f]);
                    sd = fma(m, m, sd);
                }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                sq += __shfl_xor(sq, off);
                if (BF16 || s.Csp) {
                    sh += __shfl_xor(sh, off);
                    se += __shfl_xor(se, off);
                }
                sd += __shfl_xor(sd, off);
            }
            if (lane == 0) {
                const double up = 1.0 + 1e-12;
                auto bits = [](double v) { return (unsigned long long)__double_as_longlong(v); };
                agent_store(s.cn + j, F(sq));
                if (s.cnw) s.cnw[j] = float(sq);
                if (s.cnp) {
                    uint32_t hm, l;
                    split3(float(sq), hm, l);
                    uintx4* o4 = reinterpret_cast<uintx4*>(s.cnp + int64_t(j) * 16);
                    o4[0] = uintx4{hm, l | 0x3F800000u, 0x3F803F80u, 0u};
                    o4[1] = uintx4{0u, 0u, 0u, 0u};
                }
                mx[0] = max(mx[0], bits(sqrt(sq) * up));
                if (BF16 || s.Csp) {
                    mx[1] = max(mx[1], bits(sqrt(sh) * up));
                    mx[2] = max(mx[2], bits(sqrt(se) * up + 1e-30));
                }
                if (s.cold) {
                    const double m = sqrt(sd) * up;
                    agent_store(s.drift + j, m);
                    mx[3] = max(mx[3], bits(m));
                }
            }
        }
        __syncthreads();  // the row is rewritten by the next centroid
    }
    if constexpr (BF16) {
        for (int j = k + blockIdx.x; j < s.kp; j += gridDim.x)
            for (int f = t; f < dpad; f += 256) s.Cb[int64_t(j) * dpad + f] = 0;
    }
    if (s.Cw) {
        for (int j = k + blockIdx.x; j < s.kp; j += gridDim.x) {
            for (int f = t; f < 32 * wide_chunks(d); f += 256) {
                uint16_t* o3 = s.Cw + (int64_t(f >> 5) * s.kp + j) * WIDE_ROW + (f & 31);
                for (int p = 0; p < SPLIT_PIECES; ++p) o3[32 * p] = 0;
            }
            if (t == 0) s.cnw[j] = __uint_as_float(0x7F000000u);
        }
    }
    if (s.Csp) {  // padding: zero rows with a norm of 2^127, which no threshold reaches
        for (int j = k + blockIdx.x; j < s.kp; j += gridDim.x) {
            for (int f = t; f < SPLIT_PIECES * dpad; f += 256) s.Csp[int64_t(j) * SPLIT_PIECES * dpad + f] = 0;
            if (t < 16) s.cnp[int64_t(j) * 16 + t] = t == 0 ? uint16_t(0x7F00u) : uint16_t(0);
        }
    }
    if (t == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) agent_store(s.wgmax + 4 * blockIdx.x + q, mx[q]);
    }
    if (!last_workgroup(s.ticket)) return;
    // joint maxima
    unsigned long long m[4] = {0ull, 0ull, 0ull, 0ull};
    for (int b = t; b < int(gridDim.x); b += 256)
#pragma unroll
        for (int q = 0; q < 4; ++q) m[q] = max(m[q], agent_load(s.wgmax + 4 * b + q));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int q = 0; q < 4; ++q) m[q] = max(m[q], (unsigned long long)__shfl_xor((long long)m[q], off));
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave][q] = m[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) m[q] = max(max(red[0][q], red[1][q]), max(red[2][q], red[3][q]));
    auto value = [&](int q) { return __longlong_as_double((long long)m[q]); };
    if (t < 3) s.maxima[t] = t == 0 ? value(0) : t == 1 ? value(1) : value(2);
    if constexpr (BF16) {
        const bf16_params p = make_bf16_params(value(0), value(1), value(2),
                                               __longlong_as_double((long long)s.xmax_bits[0]),
                                               __longlong_as_double((long long)s.xmax_bits[1]), s.kc);
        if (t == 0) *s.params = p;
        // cnB_j = ||c_j||^2 + B rounded up (v_j keeps its lower bound); padded ids get
        // a huge start value so they are never chosen
        for (int j = t; j < s.kp; j += 256)
            s.cnb[j] = j < k ? add_round_up(float(agent_load(s.cn + j)), float(p.B)) : __uint_as_float(0x7F000000u);
    }
    if (s.cold) {
        const double top = value(3);
        for (int j = t; j < k; j += 256) {
            const double b = (s.base[j] + (agent_load(s.drift + j) + top) * (1.0 + s.gam)) * (1.0 + 1e-15);
            s.base[j] = b < BOUND_MAX ? b : __builtin_inf();
            s.changed[j] = 0;
        }
        if (t == 0) *s.sel_count = 0;
    }
    if (t < 3) {
        if (s.acc) s.acc[t] += (unsigned long long)s.counters[t];
        s.counters[t] = 0;
    }
    if (t == 0) *s.ticket = 0u;
}

// ---------------------------------------------------------------------------
// Few rows (n <= SMALL_GROUP_ROWS, k <= SMALL_GROUP_K): the changed clusters, the
// counts, the scan and the stable grouping in one workgroup, in place of six
// launches (label_hist_kernel, sort_group_sums_kernel, scan_clusters_kernel,
// sort_block_bases_kernel, batch_scatter_kernel and the gaps between them: 24 us
// at n=10000, k=10).  Past these limits one workgroup is slower than the chip.
// Wave w takes 1/16 of the rows; ranks within a label come from one ballot per
// label bit and 64 rows, as in batch_scatter_kernel.
// ---------------------------------------------------------------------------
constexpr int SMALL_GROUP_ROWS = 16384;
constexpr int SMALL_GROUP_K = 1024;
__host__ __device__ constexpr size_t small_group_lds_bytes(int k) { return size_t(18) * k * sizeof(int32_t); }

__global__ __launch_bounds__(1024) void small_group_kernel(
    const int32_t* __restrict__ labels, int32_t* __restrict__ prev, int n, int k, int32_t* __restrict__ counts,
    int32_t* __restrict__ changed, int64_t* __restrict__ offsets, int32_t* __restrict__ chunk_base,
    int32_t* __restrict__ empty_list, int32_t* __restrict__ meta, int32_t* __restrict__ perm,
    host_report* report, const int32_t* __restrict__ open, uint32_t seq) {
    extern __shared__ int32_t glds[];
    int32_t* chg = glds + 16 * k;   // [k] members changed
    int32_t* first = chg + k;       // [k] first member position
    __shared__ int32_t sums[3][16];
    constexpr int G = SMALL_GROUP_ROWS / 1024;  // groups of 64 rows per wave
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint64_t below = (uint64_t(1) << lane) - 1u;
    int32_t* wc = glds + wave * k;
    const int per = ((n + 1023) / 1024) * 64;  // rows per wave, whole groups
    const int groups = per / 64;
    const int w0 = wave * per;
    int lbits = 0;
    while ((1 << lbits) < k) ++lbits;
    int32_t lab[G], pv[G], rk[G];
#pragma unroll
    for (int q = 0; q < G; ++q) {
        const int r = w0 + q * 64 + lane;
        const bool ok = q < groups && r < n;
        lab[q] = ok ? labels[r] : -1;
        pv[q] = ok ? prev[r] : -1;
    }
    for (int j = t; j < 17 * k; j += 1024) glds[j] = 0;  // wave counts and flags
    __syncthreads();
#pragma unroll
    for (int q = 0; q < G; ++q) {
        rk[q] = -1;
        if (q >= groups) continue;  // uniform
        const bool ok = lab[q] >= 0;
        if (ok && lab[q] != pv[q]) {
            chg[lab[q]] = 1;
            if (pv[q] >= 0) chg[pv[q]] = 1;
            prev[w0 + q * 64 + lane] = lab[q];
        }
        uint64_t same = __ballot(ok);
        for (int bit = 0; bit < lbits; ++bit) {
            const bool on = ok && ((lab[q] >> bit) & 1);
            const uint64_t m = __ballot(on);
            same &= on ? m : ~m;
        }
        const int rank = __popcll(same & below);
        if (ok) {
            rk[q] = wc[lab[q]] + rank;
            if (rank == 0) wc[lab[q]] = rk[q] + __popcll(same);
        }
    }
    __syncthreads();
    int32_t c = 0, moved = 0;
    if (t < k) {
        for (int w = 0; w < 16; ++w) {  // each wave's first position within the label
            const int32_t x = glds[w * k + t];
            glds[w * k + t] = c;
            c += x;
        }
        moved = chg[t];
        counts[t] = c;
        changed[t] = moved;
    }
    const int32_t nchk = moved ? (c + REDUCE_CHUNK - 1) / REDUCE_CHUNK : 0;
    int32_t so = c, sc = nchk, se = (t < k && c == 0) ? 1 : 0;
    scan3_1024(so, sc, se, sums);
    if (t < k) {
        offsets[t] = so - c;
        first[t] = so - c;
        chunk_base[t] = sc - nchk;
        if (c == 0) empty_list[se - 1] = t;
    }
    if (t == 1023) {
        offsets[k] = so;
        chunk_base[k] = sc;
        meta[0] = se;
        meta[1] = sc;
        report_empties(report, se, open, seq);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < G; ++q)
        if (rk[q] >= 0 && chg[lab[q]]) perm[first[lab[q]] + wc[lab[q]] + rk[q]] = w0 + q * 64 + lane;
}

}  // namespace km
