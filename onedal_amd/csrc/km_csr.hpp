// km_csr.hpp -- kernels of the CSR Lloyd path (method lloyd_csr).
//
// Replaces, on the oneDAL side (backend/gpu/kernels_csr_impl.hpp):
//   compute_data_squares            :38-55    -> csr_row_squares_kernel
//   transpose + compute_squares     :70-92, kernels_fp_impl.hpp:402-414
//                                   -> csr_transpose_kernel, csr_centroid_squares_kernel
//   assign_clusters (sparse gemm, select, complete_closest_distances)
//                                   :118-187  -> csr_assign_kernel
//   calc_objective_function         :193-203  -> csr_objective_chunks_kernel
//   update_centroids (local atomics):219-322  -> csr_chunk_sums_kernel + centroid_step_kernel
//   copy_candidates_from_data       empty_cluster_handling_dpc.cpp:152-189 -> csr_fill_empty_kernel
//
// Arithmetic (fixed order, so results are identical run to run and equal to the
// oracle's restatement; the reference's sparse gemm and atomics fix no order):
//   xs_i  = sum over the row's stored entries, in stored order, of v*v      (F)
//   cs_j  = sum_f c_jf*c_jf, features in order                              (F)
//   dot   = sum over stored entries, in stored order, of v*c_j[col]         (F, no FMA)
//   s_ij  = cs_j - 2*dot (F); label = first j with the smallest s (a NaN s_i0
//           keeps label 0, other NaNs never win); closest_i = s_i,label + xs_i (F)
//   sums  = the dense path's chunk sums (REDUCE_CHUNK members, reduce_groups
//           partials, double), adding stored entries in member order; an absent
//           entry would add +0.0, so on the same rows the sums equal the dense ones
//   objective = sum of double(closest_i) in the dense objective's order.
// Column indices need not be sorted; duplicate entries of a row are added one by
// one in stored order (sums) or overwrite in stored order (empty-cluster fill).
#pragma once

#include <type_traits>

#include "km_bounds.hpp"
#include "km_common.hpp"

namespace km {

// A workgroup's 256 rows, one per thread, walked through LDS: the rows' entries [lo, hi) are
// one run of memory, read CSR_WINDOW at a time by all threads (stage(e, p): entry p to
// slot e), then each thread takes its row's part [x, y) of the window (use), in stored
// order.  A thread reading its own row from memory touches a line per entry and lane:
// n=1e6, 20 entries a row, the three kernels that do this took 144, 90 and 124 us,
// now 36, 66 and 82 us.
constexpr int CSR_WINDOW = 4096;
template <typename Stage, typename Use>
__device__ __forceinline__ void csr_walk(int64_t lo, int64_t hi, int64_t o0, int64_t o1, Stage stage, Use use) {
    for (int64_t w0 = lo; w0 < hi; w0 += CSR_WINDOW) {
        const int cnt = int(min<int64_t>(CSR_WINDOW, hi - w0));
        __syncthreads();  // the previous window's readers are done
#pragma unroll 4
        for (int e = threadIdx.x; e < cnt; e += 256) stage(e, w0 + e);
        __syncthreads();
        const int x = int(max(o0, w0) - w0);
        const int y = int(min<int64_t>(o1 - w0, cnt));
        if (x < y) use(x, y);
    }
}

// Structure check: row offsets non-decreasing from `base` to base + nnz, every
// column index in [base, base + d).  A workgroup reads its rows' entries only after
// all their offsets passed the check.  flag bit 1: bad offsets, bit 2: bad column,
// bit 4: a row whose column indices do not increase strictly (unsorted or
// repeated; allowed, reported for the initialisation's feature-order walk and for
// the assignment's bounds).
__global__ __launch_bounds__(256) void csr_check_kernel(const int64_t* __restrict__ cols,
                                                        const int64_t* __restrict__ offs,
                                                        int64_t base, int64_t n, int64_t d,
                                                        int64_t nnz, int32_t* __restrict__ flag) {
    __shared__ int32_t sc[CSR_WINDOW];
    for (int64_t r0 = blockIdx.x * int64_t(256); r0 < n; r0 += int64_t(gridDim.x) * 256) {
        const int64_t i = r0 + threadIdx.x;
        int64_t o0 = 0, o1 = 0;
        bool ok = true;
        if (i < n) {
            o0 = offs[i] - base;
            o1 = offs[i + 1] - base;
            ok = o0 >= 0 && o1 >= o0 && o1 <= nnz;
            if (i == 0 && o0 != 0) ok = false;
            if (i == n - 1 && o1 != nnz) ok = false;
            if (!ok) atomicOr(flag, 1);
        }
        if (!__syncthreads_and(ok)) continue;
        int prev = -1;
        bool inc = true, in = true;
        csr_walk(
            offs[r0] - base, offs[min(r0 + 256, n)] - base, o0, o1,
            [&](int e, int64_t p) {
                const int64_t c = cols[p] - base;
                in = in && c >= 0 && c < d;
                sc[e] = int32_t(c);
            },
            [&](int x, int y) {
                for (int p = x; p < y; ++p) {
                    const int c = sc[p];
                    inc = inc && c > prev;
                    prev = c;
                }
            });
        if (!in) atomicOr(flag, 2);
        if (!inc) atomicOr(flag, 4);
    }
}

// xs_i: squares of a row's stored entries, summed in stored order; and (when given) the
// bits of the largest as a double (a NaN wins)
template <typename F>
__global__ __launch_bounds__(256) void csr_row_squares_kernel(const F* __restrict__ vals,
                                                              const int64_t* __restrict__ offs,
                                                              int64_t base, int64_t n,
                                                              F* __restrict__ xs,
                                                              unsigned long long* __restrict__ xmax) {
    __shared__ F sv[CSR_WINDOW];
    unsigned long long top = 0ull;
    for (int64_t r0 = blockIdx.x * int64_t(256); r0 < n; r0 += int64_t(gridDim.x) * 256) {
        const int64_t i = r0 + threadIdx.x;
        const int64_t o0 = i < n ? offs[i] - base : 0, o1 = i < n ? offs[i + 1] - base : 0;
        F acc(0);
        csr_walk(
            offs[r0] - base, offs[min(r0 + 256, n)] - base, o0, o1,
            [&](int e, int64_t p) {
                const F v = vals[p];
                sv[e] = v * v;
            },
            [&](int x, int y) {
                for (int p = x; p < y; ++p) acc = acc + sv[p];
            });
        if (i < n) {
            xs[i] = acc;
            top = max(top, (unsigned long long)__double_as_longlong(double(acc)));
        }
    }
    if (!xmax) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) top = max(top, (unsigned long long)__shfl_xor((long long)top, off));
    if ((threadIdx.x & 63) == 0) atomicMax(xmax, top);
}

// Ct (d x kp) = C^T, rows padded with zeros to kp (a multiple of the 16-byte
// vector), for coalesced vector reads over centroids: 64 x 64 tiles through LDS
// (grid: ceil(d/64) x up to 65535 workgroups of 256 threads, striding over k)
template <typename F>
__global__ __launch_bounds__(256) void csr_transpose_kernel(const F* __restrict__ C, int64_t k,
                                                            int64_t kp, int64_t d, F* __restrict__ Ct) {
    __shared__ F tile[64][65];
    const int64_t f0 = int64_t(blockIdx.x) * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int64_t j0 = int64_t(blockIdx.y) * 64; j0 < kp; j0 += int64_t(gridDim.y) * 64) {
        for (int r = ty; r < 64; r += 4) {
            const int64_t j = j0 + r, f = f0 + tx;
            if (j < k && f < d) tile[r][tx] = C[j * d + f];
        }
        __syncthreads();
        for (int r = ty; r < 64; r += 4) {
            const int64_t f = f0 + r, j = j0 + tx;
            if (j < kp && f < d) Ct[f * kp + j] = j < k ? tile[tx][r] : F(0);
        }
        __syncthreads();
    }
}

// cs_j = |c_j|^2, features in order: one wave per centroid copies the squares to LDS
// (coalesced; zeros up to a multiple of 32, which add nothing), then lane 0 adds them in
// feature order, 32 read ahead of their additions.  One serial chain of d additions.
constexpr int CSR_SQ = 32;
__host__ __device__ inline int csr_sq_len(int d) { return (d + CSR_SQ - 1) / CSR_SQ * CSR_SQ; }

template <typename F>
__global__ __launch_bounds__(64) void csr_centroid_squares_kernel(const F* __restrict__ C, int64_t k,
                                                                  int d, F* __restrict__ cs) {
    typedef F F4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(32) unsigned char sq_raw[];
    F* row = reinterpret_cast<F*>(sq_raw);  // [csr_sq_len(d)]
    const int len = csr_sq_len(d);
    for (int64_t j = blockIdx.x; j < k; j += gridDim.x) {
        for (int f = threadIdx.x; f < len; f += 64) {
            const F c = f < d ? C[j * d + f] : F(0);
            row[f] = c * c;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const F4* r4 = reinterpret_cast<const F4*>(row);
            F acc(0);
            F4 cur[CSR_SQ / 4], nxt[CSR_SQ / 4];
#pragma unroll
            for (int u = 0; u < CSR_SQ / 4; ++u) cur[u] = r4[u];
            for (int f = 0; f < len; f += CSR_SQ) {
                const int g = f + CSR_SQ < len ? f + CSR_SQ : 0;  // past the end: read, not used
#pragma unroll
                for (int u = 0; u < CSR_SQ / 4; ++u) nxt[u] = r4[g / 4 + u];
#pragma unroll
                for (int u = 0; u < CSR_SQ / 4; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc = acc + cur[u][e];
#pragma unroll
                for (int u = 0; u < CSR_SQ / 4; ++u) cur[u] = nxt[u];
            }
            cs[j] = acc;
        }
        __syncthreads();
    }
}

// value of lane u (wave-uniform u) in scalar registers
__device__ __forceinline__ float lane_value(float x, int u) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), u));
}
__device__ __forceinline__ double lane_value(double x, int u) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane(int(b & 0xFFFFFFFFll), u);
    const int hi = __builtin_amdgcn_readlane(int(b >> 32), u);
    return __longlong_as_double((long long)(unsigned(lo)) | ((long long)hi << 32));
}

__device__ __forceinline__ int64_t lane_value(int64_t x, int u) {
    const int lo = __builtin_amdgcn_readlane(int(x & 0xFFFFFFFFll), u);
    const int hi = __builtin_amdgcn_readlane(int(x >> 32), u);
    return int64_t((unsigned long long)(unsigned(lo)) | ((unsigned long long)(unsigned(hi)) << 32));
}
__device__ __forceinline__ int lane_value(int x, int u) { return __builtin_amdgcn_readlane(x, u); }

// smallest value of the wave's 64 lanes (DPP: six steps without LDS; NaN never wins)
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T dpp_from(T x) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "lane values");
    if constexpr (sizeof(T) == 4) {
        const int v = __builtin_bit_cast(int, x);
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xf, false));
    } else {
        const long long v = __builtin_bit_cast(long long, x);
        const int lo = int(v & 0xFFFFFFFFll), hi = int(v >> 32);
        const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
        const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
        return __builtin_bit_cast(T, (long long)(unsigned(l2)) | ((long long)h2 << 32));
    }
}
__device__ __forceinline__ float lower(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ double lower(double a, double b) { return fmin(a, b); }
__device__ __forceinline__ int lower(int a, int b) { return min(a, b); }
__device__ __forceinline__ float higher(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double higher(double a, double b) { return fmax(a, b); }
template <typename T>
__device__ __forceinline__ T wave_lowest(T x) {
    x = lower(x, dpp_from<0x111, 0xf>(x));  // row_shr 1, 2, 4, 8: lane 15 of each row of 16
    x = lower(x, dpp_from<0x112, 0xf>(x));
    x = lower(x, dpp_from<0x114, 0xf>(x));
    x = lower(x, dpp_from<0x118, 0xf>(x));
    x = lower(x, dpp_from<0x142, 0xa>(x));  // row_bcast 15, 31: lane 63
    x = lower(x, dpp_from<0x143, 0xc>(x));
    return lane_value(x, 63);
}
// the same steps as one instruction each (the compiler's form takes five: a copy, the
// move, and two operands made canonical); a DPP operand is read two cycles after a write
template <>
__device__ __forceinline__ float wave_lowest<float>(float x) {
    asm("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(x));
    return lane_value(x, 63);
}

// 16-byte vectors of F
template <typename F>
struct csr_vec;
template <>
struct csr_vec<float> {
    static constexpr int N = 4;
    typedef float type __attribute__((ext_vector_type(4)));
};
template <>
struct csr_vec<double> {
    static constexpr int N = 2;
    typedef double type __attribute__((ext_vector_type(2)));
};

// (s, j) candidate order: the smaller s wins, equal values go to the lower j;
// NaN never wins (has == false stands for "no candidate yet")
template <typename F>
__device__ __forceinline__ void csr_take(F& bs, int& bj, bool& has, F s, int j) {
    if (s != s) return;
    if (!has || s < bs || (s == bs && j < bj)) {
        bs = s;
        bj = j;
        has = true;
    }
}

// Bounds (km_bounds.hpp) for rows whose columns increase strictly (so that the stored
// entries are a vector).  The label is the smallest computed s_ij, whose error is
//     |s_ij - (||c_j||^2 - 2 x.c_j)| <= g (||c_j||^2 + 2 ||x|| ||c_j||) <= 3 g M^2,
// g = gamma_{d+4} and M the largest norm of a row or centroid: not relative to the
// distance, as the dense form's.  With d_j - d_a >= G > 0 for every other centroid,
// d_j^2 - d_a^2 >= G^2, so a row stays settled while G > sqrt(2 * 3 g M^2): that part is
// taken off its gap when it is settled.  M may be taken at that time: later centroids
// are means of rows, rows, or unchanged.
struct csr_bounds {
    const unsigned long long* xmax;  // csr_row_squares_kernel
    const double* cmax;              // max ||c_j||, rounded up
    double g;                        // gamma_{d+4}
};

// gap of a row settled with the smallest s (best) and the next one (second, a float at most
// as large; the wave's lowest float takes a fifth of the instructions of a double), xs its squares;
// loose: band's worth of rounding in best besides its own
__device__ __forceinline__ float csr_gap(double best, double second, double xs, double band, double loose,
                                         const row_select& rs, int lab) {
    if (!(band < BOUND_MAX) || best != best) return -__builtin_inff();
    const float g = bound_gap(best + xs + (4.5 + loose) * band, second - 4.5 * band + xs, rs.gam, rs.base[lab]);
    return float_below(double(g) - sqrt(6.3 * band));
}
// g M^2
__device__ __forceinline__ double csr_band(const csr_bounds& kb) {
    const double C = *kb.cmax;
    const double M = fmax(sqrt(__longlong_as_double((long long)*kb.xmax)) * (1.0 + kb.g), C) * (1.0 + 1e-6);
    return M < BOUND_MAX && C < BOUND_MAX ? kb.g * M * M : __builtin_inf();  // NaN as well
}

// The dots where csr_assign_kernel's runs of rows are slower: transposed centroids past an
// XCD's L2, or more than 128 VEC of them.
// One wave per row.  Lane l accumulates the dots of the VEC consecutive
// centroids jb + VEC (l + 64 t) + e (t < JT, e < VEC) over the row's entries,
// which are loaded 64 at a time and taken in stored order from their lanes;
// each entry reads one 16-byte vector of its transposed-centroid row per t.  Few
// registers, so that eight waves a SIMD hide the reads, which miss the L2 here: k = 500, d = 4000,
// n=3e5, 40 entries takes 1.51 ms, 1.68 ms with runs of rows (double: 2.8 and 5.0), 2.05 with
// a lane's four reads issued together.
// Then each lane's best and a wave reduction (ties to the lower j).  BND: the rows of rs,
// and the second best of each, from which csr_gap_kernel forms the gaps (3.3 ms a pass in
// double for the same rows).
template <typename F, bool BND>
__global__ __launch_bounds__(256, 8) void csr_assign_blocks_kernel(
    const F* __restrict__ vals, const int64_t* __restrict__ cols, const int64_t* __restrict__ offs,
    int64_t base, int64_t n, int k, int kp, const F* __restrict__ Ct, const F* __restrict__ cs,
    const F* __restrict__ xs, int32_t* __restrict__ labels, F* __restrict__ closest, row_select rs,
    float* __restrict__ second) {
    constexpr int VEC = csr_vec<F>::N;
    constexpr int JT = 4;
    typedef typename csr_vec<F>::type V;
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = (int64_t(gridDim.x) * blockDim.x) >> 6;
    const int64_t nsel = BND ? select_rows(rs, n) : n;
    for (int64_t r = wave; r < nsel; r += nwaves) {
        const int64_t i = BND ? select_row(rs, r) : r;
        const int64_t o0 = offs[i] - base, o1 = offs[i + 1] - base;
        F bs = fp_traits<F>::inf, b2 = fp_traits<F>::inf;
        int bj = 0;
        bool has = false;
        F s0(0);  // s of centroid 0 (lane 0, first block)
        for (int jb = 0; jb < k; jb += 64 * VEC * JT) {
            F acc[JT][VEC];
#pragma unroll
            for (int t = 0; t < JT; ++t)
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[t][e] = F(0);
            for (int64_t p0 = o0; p0 < o1; p0 += 64) {
                const int cnt = int(min<int64_t>(64, o1 - p0));
                int my_c = 0;  // a column index (< d <= 4096)
                F my_v(0);
                if (lane < cnt) {
                    my_c = int(cols[p0 + lane] - base);
                    my_v = vals[p0 + lane];
                }
                for (int u = 0; u < cnt; ++u) {
                    // entry u of the group, read from its lane into scalar registers
                    const int c = __builtin_amdgcn_readlane(my_c, u);
                    const F v = lane_value(my_v, u);
                    const F* crow = Ct + int64_t(c) * kp;
#pragma unroll
                    for (int t = 0; t < JT; ++t) {
                        const int j = jb + VEC * (64 * t + lane);
                        if (j < k) {
                            const V cv = *reinterpret_cast<const V*>(crow + j);
#pragma unroll
                            for (int e = 0; e < VEC; ++e) {
                                const F pr = v * cv[e];
                                acc[t][e] = acc[t][e] + pr;
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < JT; ++t)
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const int j = jb + VEC * (64 * t + lane) + e;
                    if (j < k) {
                        const F two_dot = F(2) * acc[t][e];
                        const F s = cs[j] - two_dot;
                        if (j == 0) s0 = s;
                        // ascending j in a lane: an equal value is the later one; bs is
                        // infinite before the first.  A NaN only lowers b2.
                        if (BND) b2 = lower(b2, higher(bs, s));
                        const bool win = s < bs || (!has && s == s);
                        bs = win ? s : bs;
                        bj = win ? j : bj;
                        has = has || win;
                    }
                }
        }
        const F mine = bs;
        const int my_j = bj;
        const bool mine_has = has;
        // wave reduction of (bs, bj, has)
        for (int off = 32; off > 0; off >>= 1) {
            const F os = __shfl_xor(bs, off);
            const int oj = __shfl_xor(bj, off);
            const int oh = __shfl_xor(int(has), off);
            if (oh) csr_take(bs, bj, has, os, oj);
        }
        s0 = __shfl(s0, 0);
        if (lane == 0) {
            int lab = bj;
            F best = bs;
            if (s0 != s0 || !has) {  // s_i0 NaN, or every s NaN: label 0
                lab = 0;
                best = s0;
            }
            labels[i] = lab;
            closest[i] = best + xs[i];
        }
        if (BND) {
            const float s2 = wave_lowest(!mine_has ? __builtin_inff() : float_below(double(my_j == bj ? b2 : mine)));
            if (lane == 0) second[i] = s2;
        }
    }
}

// the gaps after csr_assign_blocks_kernel, a thread per row: there they would cost a whole
// wave's instructions.  best comes back from closest, which rounds twice.
template <typename F>
__global__ __launch_bounds__(256) void csr_gap_kernel(int64_t n, const F* __restrict__ xs,
                                                      const F* __restrict__ closest, const float* __restrict__ second,
                                                      const int32_t* __restrict__ labels, row_select rs,
                                                      csr_bounds kb) {
    const double band = csr_band(kb);
    const int64_t nsel = select_rows(rs, n);
    for (int64_t e = blockIdx.x * int64_t(256) + threadIdx.x; e < nsel; e += int64_t(gridDim.x) * 256) {
        const int64_t i = select_row(rs, e);
        rs.gap[i] = csr_gap(double(closest[i]) - double(xs[i]), double(second[i]), double(xs[i]), band, 1.0, rs, labels[i]);
    }
}

// reads through a buffer descriptor: a lane's byte offset and the wave's, no 64-bit address
// arithmetic
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
template <typename V>
__device__ __forceinline__ V buffer_read(__amdgpu_buffer_rsrc_t r, int lane_off, int wave_off) {
    if constexpr (sizeof(V) == 4)
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, lane_off, wave_off, 0));
    else if constexpr (sizeof(V) == 8)
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, wave_off, 0));
    else
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, wave_off, 0));
}

// Rows are taken in runs of up to 16 per wave (their offsets read and their results written
// together, by lanes), one wave per row.  Lane l accumulates the dots of the VEC consecutive
// centroids VEC (l + 64 t) + e (t < JT, e < VEC: one block holds k) over the row's entries,
// which are loaded 64 at a time (a row's first ones during the row before) and taken in
// stored order from their lanes; each entry reads one 16-byte vector of its
// transposed-centroid row per t, U in flight.  Then each lane's best and a wave
// reduction (ties to the lower j).
//
// BND: the rows of rs, and the second best as well, for the gap of each.
//
// Taken for k up to 128 VEC and transposed centroids up to an XCD's L2 (n=1e6, d=2000, 20
// entries, k=256 in double, 4 MB: 1.79 ms, 2.29 with a row per wave at a time; past it
// csr_assign_blocks_kernel is the faster one).
// Bound by a row's instructions, not by bytes (more reads in flight changed nothing): n=1e6, 20
// entries, k=256 1.3 ms for all rows.  Dots from a half-precision copy of the centroids
// first, the others where those left several, took 0.8-1.0 ms, but held the centroids in 16
// bits, and rows in random columns (n=1e5, 50 entries, k=256) paid for both: 8 iterations
// to a threshold 4.2 ms, 3.9 ms without.
constexpr int64_t CSR_RUNS_BYTES = int64_t(4) << 20;
template <typename F, int JT, bool BND>
__global__ __launch_bounds__(256) void csr_assign_kernel(
    const F* __restrict__ vals, const int64_t* __restrict__ cols, const int64_t* __restrict__ offs,
    int64_t base, int64_t n, int d, int k, int kp, const F* __restrict__ Ct, const F* __restrict__ cs,
    const F* __restrict__ xs, int32_t* __restrict__ labels, F* __restrict__ closest, row_select rs, csr_bounds kb) {
    constexpr int VEC = csr_vec<F>::N;
    constexpr int U = 8 / JT;  // entries whose vectors are in flight together
    typedef typename csr_vec<F>::type V;
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = (int64_t(gridDim.x) * blockDim.x) >> 6;
    const int64_t nsel = BND ? select_rows(rs, n) : n;
    const int per = int(max<int64_t>(1, min<int64_t>(16, nsel / nwaves)));
    const int64_t nruns = (nsel + per - 1) / per;
    const double band = BND ? csr_band(kb) : 0.0;
    // (at most CSR_RUNS_BYTES)
    const auto rsrc = buffer_of(Ct, int(int64_t(sizeof(F)) * d * kp));
    F csv[JT][VEC];  // the same for every row
    int off[JT];     // a lane past k reads the last vector, for nothing
#pragma unroll
    for (int t = 0; t < JT; ++t) {
        off[t] = min(VEC * (64 * t + lane), kp - VEC) * int(sizeof(F));
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const int j = VEC * (64 * t + lane) + e;
            csv[t][e] = j < k ? cs[j] : F(0);
        }
    }
    for (int64_t run = wave; run < nruns; run += nwaves) {
        const int64_t e0 = run * per;
        const int rows = int(min<int64_t>(per, nsel - e0));
        // lane q holds row q of the run, and its results
        int64_t my_row = 0, my_o0 = 0, my_o1 = 0;
        F my_xs(0), my_best(0);
        float my_second = __builtin_inff();
        int my_lab = 0;
        if (lane < rows) {
            my_row = BND ? select_row(rs, e0 + lane) : e0 + lane;
            my_o0 = offs[my_row] - base;
            my_o1 = offs[my_row + 1] - base;
            my_xs = xs[my_row];
        }
        auto fetch = [&](int64_t p0, int64_t o1, int& c, F& v) {
            c = 0;  // the byte offset of a column's row of Ct
            v = F(0);
            if (p0 + lane < o1) {
                c = int(cols[p0 + lane] - base) * kp * int(sizeof(F));
                v = vals[p0 + lane];
            }
        };
        int next_c;
        F next_v;
        fetch(lane_value(my_o0, 0), lane_value(my_o1, 0), next_c, next_v);
        for (int q = 0; q < rows; ++q) {
            const int64_t o0 = lane_value(my_o0, q), o1 = lane_value(my_o1, q);
            const int first_c = next_c;
            const F first_v = next_v;
            if (q + 1 < rows) fetch(lane_value(my_o0, q + 1), lane_value(my_o1, q + 1), next_c, next_v);
            F acc[JT][VEC];
#pragma unroll
            for (int t = 0; t < JT; ++t)
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[t][e] = F(0);
            // entries u0 .. of the 64 held, the first `left` of a group
            auto add = [&](int c_of, F v_of, int u0, int left, auto count) {
                constexpr int N = decltype(count)::value;
                V cv[N][JT];
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const int at = lane_value(c_of, u0 + u);
#pragma unroll
                    for (int t = 0; t < JT; ++t) cv[u][t] = buffer_read<V>(rsrc, off[t], at);
                }
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const F v = lane_value(v_of, u0 + u);
                    if (u >= left) break;  // nothing added: a centroid may be infinite
#pragma unroll
                    for (int t = 0; t < JT; ++t)
#pragma unroll
                        for (int e = 0; e < VEC; ++e) {
                            const F pr = v * cv[u][t][e];
                            acc[t][e] = acc[t][e] + pr;
                        }
                }
            };
            for (int64_t p0 = o0; p0 < o1; p0 += 64) {
                const int cnt = int(min<int64_t>(64, o1 - p0));
                int my_c = first_c;
                F my_v = first_v;
                if (p0 != o0) fetch(p0, o1, my_c, my_v);
                // whole groups, then the smallest group that holds the rest: past the
                // last entry the column is 0, and add() leaves the value out
                int u = 0;
                for (; cnt - u > U / 2; u += U) add(my_c, my_v, u, cnt - u, std::integral_constant<int, U>());
                if (cnt - u > U / 4) add(my_c, my_v, u, cnt - u, std::integral_constant<int, U / 2>());
                else if (cnt > u) add(my_c, my_v, u, cnt - u, std::integral_constant<int, U / 4>());
            }
            F bs(0), b2 = fp_traits<F>::inf;  // best and second best of this lane
            int bj = 0;
            bool has = false;
            F s0(0);  // s of centroid 0 (lane 0)
#pragma unroll
            for (int t = 0; t < JT; ++t)
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const int j = VEC * (64 * t + lane) + e;
                    const F two_dot = F(2) * acc[t][e];
                    const F s = csv[t][e] - two_dot;
                    if (j == 0) s0 = s;
                    // ascending j in a lane: an equal value is the later one
                    const bool in = j < k && s == s;
                    const bool win = in && (!has || s < bs);
                    if (BND && in) b2 = win ? (has ? bs : b2) : lower(b2, s);
                    bs = win ? s : bs;
                    bj = win ? j : bj;
                    has = has || win;
                }
            // the smallest s, then the lowest j that has it; every s NaN, or s_i0: label 0
            const F best = wave_lowest(has ? bs : fp_traits<F>::inf);
            const int lab = wave_lowest(has && bs == best ? bj : 0x7fffffff);
            s0 = lane_value(s0, 0);
            const bool none = lab == 0x7fffffff || s0 != s0;
            float second = __builtin_inff();
            if (BND) second = wave_lowest(!has ? __builtin_inff() : float_below(double(bj == lab ? b2 : bs)));
            if (lane == q) {
                my_lab = none ? 0 : lab;
                my_best = none ? s0 : best;
                my_second = second;
            }
        }
        if (lane < rows) {
            labels[my_row] = my_lab;
            closest[my_row] = my_best + my_xs;
            if (BND)
                rs.gap[my_row] = csr_gap(double(my_best), double(my_second), double(my_xs), band, 0.0, rs, my_lab);
        }
    }
}

// closest_i of rows with their label known: the arithmetic of csr_assign_kernel for one
// centroid, a lane per row.  With gap, of the settled rows alone (bound_select_kernel's
// test), which the next assignment leaves out: an assigned row gets its closest there.
template <typename F>
__global__ __launch_bounds__(256) void csr_closest_kernel(
    const F* __restrict__ vals, const int64_t* __restrict__ cols, const int64_t* __restrict__ offs, int64_t base,
    int64_t n, int d, const F* __restrict__ C, const F* __restrict__ cs, const F* __restrict__ xs,
    const int32_t* __restrict__ labels, F* __restrict__ closest, const float* __restrict__ gap,
    const double* __restrict__ bound) {
    constexpr int U = 8;  // gathers in flight
    __shared__ int32_t sc[CSR_WINDOW];
    __shared__ F sv[CSR_WINDOW];
    for (int64_t r0 = blockIdx.x * int64_t(256); r0 < n; r0 += int64_t(gridDim.x) * 256) {
        const int64_t i = r0 + threadIdx.x;
        const int lab = i < n ? labels[i] : 0;
        const bool mine = i < n && (!gap || double(gap[i]) > bound[lab] + BOUND_SLACK);
        if (!__syncthreads_or(mine)) continue;
        const int64_t o0 = mine ? offs[i] - base : 0, o1 = mine ? offs[i + 1] - base : 0;
        const F* c = C + int64_t(lab) * d;
        F acc(0);
        csr_walk(
            offs[r0] - base, offs[min(r0 + 256, n)] - base, o0, o1,
            [&](int e, int64_t p) {
                sc[e] = int32_t(cols[p] - base);
                sv[e] = vals[p];
            },
            [&](int x, int y) {
                for (int p = x; p < y; p += U) {
                    F v[U], w[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int q = min(p + u, y - 1);
                        v[u] = sv[q];
                        w[u] = c[sc[q]];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const F pr = v[u] * w[u];
                        const F t = acc + pr;
                        acc = p + u < y ? t : acc;
                    }
                }
            });
        if (mine) {
            const F two_dot = F(2) * acc;
            const F s = cs[lab] - two_dot;
            closest[i] = s + xs[i];
        }
    }
}

// objective over closest_i (as double) in the dense objective's order; also
// writes the per-row keys used to pick empty-cluster candidates (and subtracted
// from the objective for each one taken)
template <typename F>
__global__ __launch_bounds__(256) void csr_objective_chunks_kernel(const F* __restrict__ closest,
                                                                   int64_t n,
                                                                   double* __restrict__ d64_out,
                                                                   double* __restrict__ chunk_sums) {
    __shared__ double part[256];
    const int t = threadIdx.x;
    const int64_t nchunks = (n + OBJ_CHUNK - 1) / OBJ_CHUNK;
    for (int64_t q = blockIdx.x; q < nchunks; q += gridDim.x) {
        const int64_t r0 = q * OBJ_CHUNK;
        const int rows = int(min<int64_t>(OBJ_CHUNK, n - r0));
        double p = 0.0;
        for (int r = t; r < rows; r += 256) {
            const double v = double(closest[r0 + r]);
            // candidate keys: a rounding-negative distance counts as 0 (the
            // radix select orders the raw bits, which is numeric only for +0 and up)
            if (d64_out) d64_out[r0 + r] = (v != v || v > 0.0) ? v : 0.0;
            p = p + v;
        }
        part[t] = p;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (t < s) part[t] = part[t] + part[t + s];
            __syncthreads();
        }
        if (t == 0) chunk_sums[q] = part[0];
        __syncthreads();
    }
}

// members whose entries are loaded together by the chunk-sum kernel
constexpr int CSR_AHEAD = 8;

// *p += v in LDS.  float: one ds_add_f64 (sums of floats are never denormal doubles, so no
// mode changes their bits), which the next member's add does not wait for as it waits
// for a read and a write
__device__ __forceinline__ void csr_add(double* p, float v) {
    __hip_atomic_fetch_add(p, double(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void csr_add(double* p, double v) { *p = *p + v; }

// Chunk sums of the CSR rows: one single-wave workgroup per chunk of
// REDUCE_CHUNK members, G = reduce_groups(d) partial vectors of d doubles in LDS
// (member m of the chunk goes to partial m % G).  A row whose column indices are
// strictly increasing is added by all lanes at once (distinct columns); any
// other row by lane 0 alone, entry by entry, so every column is summed in member
// order and, inside a row, in stored order.  Partials are added in g order.
// The wave's LDS operations execute in issue order, so a member's adds see the
// previous member's.  Groups of 64 members whose rows all hold at most 64
// entries load CSR_AHEAD rows' entries at a time into registers (the offsets of
// the whole group first), the next ones while these are added; other groups go member
// by member.  INC: every row's columns are known to increase, nothing is compared.
// n=1e6, 20 entries, d=2000: 304 us for all rows, 340 us with the comparison and
// without the loads ahead.
template <typename F, bool INC>
__global__ __launch_bounds__(64) void csr_chunk_sums_kernel(
    const F* __restrict__ vals, const int64_t* __restrict__ cols, const int64_t* __restrict__ offs,
    int64_t base, int d, int k, const int32_t* __restrict__ perm,
    const int64_t* __restrict__ offsets, const int32_t* __restrict__ chunk_base,
    const int32_t* __restrict__ meta, double* __restrict__ part) {
    extern __shared__ double acc[];  // [G * d]
    const int lane = threadIdx.x;
    const int total = meta[1];
    const int G = reduce_groups(d);
    const int width = G * d;
    for (int q = blockIdx.x; q < total; q += gridDim.x) {
        int lo = 0, hi = k;  // chunk_base[k] = total > q
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (chunk_base[mid] <= q) lo = mid; else hi = mid;
        }
        const int j = lo;
        const int64_t m_begin = offsets[j] + int64_t(q - chunk_base[j]) * REDUCE_CHUNK;
        const int64_t m_end = min(m_begin + REDUCE_CHUNK, offsets[j + 1]);
        for (int e = lane; e < width; e += 64) acc[e] = 0.0;
        __syncthreads();
        // groups of up to 64 members: lane t holds member t's row and offsets
        for (int64_t m0 = m_begin; m0 < m_end; m0 += 64) {
            const int cnt = int(min<int64_t>(64, m_end - m0));
            int64_t my_o0 = 0;
            int my_len = 0;
            if (lane < cnt) {
                const int64_t row = perm[m0 + lane];
                my_o0 = offs[row] - base;
                my_len = int(offs[row + 1] - base - my_o0);
            }
            if (__all(my_len <= 64)) {
                // every row fits the lanes: the entries of CSR_AHEAD members are
                // loaded together, then added member by member
                int cc[2][CSR_AHEAD];
                F vv[2][CSR_AHEAD];
                auto load = [&](int u0, int (&c)[CSR_AHEAD], F (&v)[CSR_AHEAD]) {
#pragma unroll
                    for (int q = 0; q < CSR_AHEAD; ++q) {
                        const int m = min(u0 + q, cnt - 1);
                        const int64_t o0 = lane_value(my_o0, m);
                        c[q] = 0;
                        v[q] = F(0);
                        if (lane < __builtin_amdgcn_readlane(my_len, m)) {
                            c[q] = int(cols[o0 + lane] - base);
                            v[q] = vals[o0 + lane];
                        }
                    }
                };
                auto add = [&](int u0, const int (&c)[CSR_AHEAD], const F (&v)[CSR_AHEAD]) {
#pragma unroll
                    for (int q = 0; q < CSR_AHEAD; ++q) {
                        if (u0 + q >= cnt) break;  // uniform
                        const int len = __builtin_amdgcn_readlane(my_len, u0 + q);
                        double* pg = acc + int((m0 + u0 + q - m_begin) % G) * d;
                        bool inc = true;
                        if (!INC) {
                            const int prev = __shfl_up(c[q], 1);
                            inc = __all(lane == 0 || lane >= len || prev < c[q]);
                        }
                        if (inc) {
                            // strictly increasing columns: distinct, added at once
                            if (lane < len) csr_add(pg + c[q], v[q]);
                        } else {
                            for (int e = 0; e < len; ++e) {
                                const int ce = __builtin_amdgcn_readlane(c[q], e);
                                const F ve = lane_value(v[q], e);
                                if (lane == 0) pg[ce] = pg[ce] + double(ve);
                            }
                        }
                    }
                };
                load(0, cc[0], vv[0]);
                for (int u0 = 0; u0 < cnt; u0 += 2 * CSR_AHEAD) {
                    if (u0 + CSR_AHEAD < cnt) load(u0 + CSR_AHEAD, cc[1], vv[1]);
                    add(u0, cc[0], vv[0]);
                    if (u0 + CSR_AHEAD >= cnt) break;
                    if (u0 + 2 * CSR_AHEAD < cnt) load(u0 + 2 * CSR_AHEAD, cc[0], vv[0]);
                    add(u0 + CSR_AHEAD, cc[1], vv[1]);
                }
                continue;
            }
            for (int64_t m = m0; m < m0 + cnt; ++m) {
                const int64_t row = perm[m];
                double* pg = acc + int((m - m_begin) % G) * d;
                const int64_t o0 = offs[row] - base, o1 = offs[row + 1] - base;
                bool sorted = true;
                for (int64_t p = o0 + 1 + lane; p < o1; p += 64)
                    if (cols[p] <= cols[p - 1]) sorted = false;
                sorted = __all(sorted);
                if (sorted) {
                    for (int64_t p = o0 + lane; p < o1; p += 64) {
                        const int64_t c = cols[p] - base;
                        pg[c] = pg[c] + double(vals[p]);
                    }
                } else if (lane == 0) {
                    for (int64_t p = o0; p < o1; ++p) {
                        const int64_t c = cols[p] - base;
                        pg[c] = pg[c] + double(vals[p]);
                    }
                }
                __syncthreads();
            }
        }
        for (int f = lane; f < d; f += 64) {
            double t = acc[f];
            for (int g = 1; g < G; ++g) t = t + acc[g * d + f];
            part[int64_t(q) * d + f] = t;
        }
        __syncthreads();
    }
}

// empty cluster e takes candidate row cand[e]: zeros, then the stored entries in
// stored order (a later duplicate overwrites)
template <typename F>
__global__ __launch_bounds__(64) void csr_fill_empty_kernel(
    const F* __restrict__ vals, const int64_t* __restrict__ cols, const int64_t* __restrict__ offs,
    int64_t base, int d, const int32_t* __restrict__ empty_list, const int32_t* __restrict__ cand,
    const int32_t* __restrict__ meta, F* __restrict__ Cnext) {
    const int m = meta[0];  // empty clusters this iteration (picks in cand, ec_order_kernel)
    for (int e = blockIdx.x; e < m; e += gridDim.x) {
        F* dst = Cnext + int64_t(empty_list[e]) * d;
        for (int f = threadIdx.x; f < d; f += blockDim.x) dst[f] = F(0);
        __syncthreads();
        if (threadIdx.x == 0) {
            const int64_t row = cand[e];
            const int64_t o0 = offs[row] - base, o1 = offs[row + 1] - base;
            for (int64_t p = o0; p < o1; ++p) dst[cols[p] - base] = vals[p];
        }
        __syncthreads();
    }
}

}  // namespace km
