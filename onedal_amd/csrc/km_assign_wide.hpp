// km_assign_wide.hpp -- FP32 assignment of wide rows (d > 128) on the BF16 matrix cores.
//
// The split products and the error band of km_assign_split.hpp, for rows whose halves do
// not fit a wave's registers: a tiled product over chunks of 32 features.  It replaces
// a VALU tile kernel for d > 256 (n=1e5, d=512, k=256: 0.64 ms a pass over all rows, now
// 0.14 ms; ten iterations 7.1 -> 3.6 ms) and the FP32 matrix-core kernel for
// 128 < d <= 256 (inference of n=1e6, d=200, k=300: 2.27 -> 0.99 ms).
//
// Workgroup = 2 x NWC waves on a tile of 128 rows x 64 NWC centroids; a wave owns 64 x 64
// (two row blocks, two centroid blocks, 64 accumulators a lane).  Per chunk a row is
// one full 128-byte line of X, read by eight lanes, split into its bf16 halves once
// and staged in LDS beside the centroids' chunk (both halves, laid out chunk by
// chunk by the centroid step, so a tile's chunk is one contiguous run): 128 bytes a
// row and chunk, 16-byte vector q of row r at q ^ (r & 7).  Two buffers; the next chunk's
// loads (rows: two chunks ahead, they come from HBM) are in flight during the
// products.  NWC = 4 reads the rows once for k <= 256 (one workgroup of 8 waves per
// CU); NWC = 2, for k <= 128, leaves no wave on padding and fits twice.
// Bound: per chunk a wave's 24 products take 768 cycles and its LDS reads 16 KB, about
// the same time at two waves per SIMD.
//
// Error bound: as in km_assign_split.hpp, but each chunk's small products meet the sum
// of the chunks before, so the whole chain of 3 d additions is bounded against
// 2.04 X C (gamma_3d instead of gamma_d).
//
// The norms are added after the products: v_j = (acc + s) + ||c_j||^2, s = ||x||^2 + the
// band's error (rounded up), so the values are positive and keys order like them.  Every
// lane keeps a top-2 slot per (row block, centroid block); a row's 4 NWC slots meet in
// LDS after the last centroid tile and one thread settles the row.
#pragma once

#include "km_assign_split.hpp"

namespace km {

constexpr int WIDE_ROWS = 128;
// relative error of ||x||^2: chains of d / 8 <= 512 additions (the engine takes d <= 4096)
// and three more
constexpr float WIDE_NORM_UP = 3.3e-5f;
__host__ __device__ constexpr int wide_cols(int nwc) { return 64 * nwc; }
// bytes of the centroid operand: kp rows x whole chunks of 32 features x two halves
__host__ inline int wide_kp(int k, int nwc) { return (k + wide_cols(nwc) - 1) / wide_cols(nwc) * wide_cols(nwc); }
__host__ __device__ inline int wide_chunks(int d) { return (d + 31) / 32; }
__host__ inline size_t wide_lds_bytes(int nwc) { return size_t(2) * 128 * (wide_cols(nwc) + WIDE_ROWS); }

// Cw: [chunk][kp][hi 32 | lo 32] bf16 of -2 c; cnw: kp values ||c_j||^2 (padding: huge)
template <int NWC>
__global__ __launch_bounds__(128 * NWC, 2) void assign_wide_kernel(
    const float* __restrict__ X, int64_t n, int d, const uint16_t* __restrict__ Cw, const float* __restrict__ cnw,
    int k, int kp, const double* __restrict__ cmax_p, split_consts kc, int32_t* __restrict__ labels,
    refine_lists L, row_select rs) {
    constexpr int T = 128 * NWC;            // threads
    constexpr int COLS = wide_cols(NWC);
    constexpr int XV = WIDE_ROWS * 8 / T;   // 16-byte vectors of X per thread and chunk
    constexpr int CV = COLS * 8 / T;        // of the centroid operand
    constexpr int NSLOT = 4 * NWC;          // slots of a row: NWC waves x 2 blocks x 2 halves
    extern __shared__ __align__(16) unsigned char smem_raw[];
    unsigned char* Cbuf = smem_raw;                       // [2][COLS][128]
    unsigned char* Xbuf = smem_raw + 2 * COLS * 128;      // [2][WIDE_ROWS][128]
    __shared__ float rx2[WIDE_ROWS], rs_s[WIDE_ROWS], rda[WIDE_ROWS];
    __shared__ int32_t rrow[WIDE_ROWS];
    __shared__ int open_cnt[2], open_base[2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / NWC, wc = wave % NWC;  // row half and column quarter of the wave
    const int r32 = lane & 31, h = lane >> 5;
    const float C = float(*cmax_p) * (1.0f + 2.4e-7f);
    const uint32_t kmask = 0x7FFFFFFFu & ~((1u << kc.ib) - 1u);
    const int chunks = wide_chunks(d);
    const int ctiles = kp / COLS;
    const int64_t nsel = select_rows(rs, n);
    const int64_t ntiles = (nsel + WIDE_ROWS - 1) / WIDE_ROWS;
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t n0 = tile * WIDE_ROWS;
        __syncthreads();  // the previous tile's readers are done
        if (tid < WIDE_ROWS) rrow[tid] = n0 + tid < nsel ? int32_t(select_row(rs, n0 + tid)) : -1;
        if (tid < 2) open_cnt[tid] = 0;
        __syncthreads();
        // this thread's vectors: row tid / 8 + i T / 8, vector tid % 8 of each chunk
        const float* xsrc[XV];
        int64_t xav[XV];  // floats from xsrc to the end of X (0: no row)
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            const int row = rrow[(tid >> 3) + i * (T / 8)];
            xsrc[i] = X + int64_t(row < 0 ? 0 : row) * d + 4 * (tid & 7);
            xav[i] = row < 0 ? 0 : (n - row) * d - 4 * (tid & 7);
        }
        const int xleft = d - 4 * (tid & 7);  // features from this thread's vector on
        auto load_x = [&](int c, floatx4(&v)[XV]) {
#pragma unroll
            for (int i = 0; i < XV; ++i) {
                floatx4 t = {0.f, 0.f, 0.f, 0.f};
                const int f = 32 * c;
                if (f < xleft && xav[i] > 0) {
                    if (f + 4 <= xav[i]) {
                        t = *reinterpret_cast<const floatx4u*>(xsrc[i] + f);
                    } else {
                        t[0] = xsrc[i][f];
                        if (f + 1 < xleft) t[1] = xsrc[i][f + 1];
                        if (f + 2 < xleft) t[2] = xsrc[i][f + 2];
                    }
                }
                v[i] = t;
            }
        };
        auto load_c = [&](int ct, int c, uintx4(&v)[CV]) {
            const uintx4* src = reinterpret_cast<const uintx4*>(Cw + (int64_t(c) * kp + int64_t(ct) * COLS) * 64);
#pragma unroll
            for (int i = 0; i < CV; ++i) v[i] = src[tid + i * T];
        };
        float sq[XV];
#pragma unroll
        for (int i = 0; i < XV; ++i) sq[i] = 0.f;
        auto store_x = [&](int c, int b, floatx4(&v)[XV], bool norms) {
#pragma unroll
            for (int i = 0; i < XV; ++i) {
                const int r = (tid >> 3) + i * (T / 8), q = tid & 7;  // features 4 q .. of the chunk
                floatx4 x = v[i];
                if (d & 3) {
#pragma unroll
                    for (int u = 1; u < 4; ++u) x[u] = 32 * c + u < xleft ? x[u] : 0.f;
                }
                if (norms) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) sq[i] = __builtin_fmaf(x[u], x[u], sq[i]);
                }
                uint32_t h0, l0, h1, l1;
                split2(x[0], x[1], h0, l0);
                split2(x[2], x[3], h1, l1);
                unsigned char* base = Xbuf + (b * WIDE_ROWS + r) * 128;
                const int o = (q & 1) * 8;
                *reinterpret_cast<uint2*>(base + (((q >> 1) ^ (r & 7)) * 16) + o) = make_uint2(h0, h1);
                *reinterpret_cast<uint2*>(base + (((4 + (q >> 1)) ^ (r & 7)) * 16) + o) = make_uint2(l0, l1);
            }
        };
        auto store_c = [&](int b, uintx4(&v)[CV]) {
#pragma unroll
            for (int i = 0; i < CV; ++i) {
                const int e = tid + i * T, r = e >> 3, q = e & 7;
                *reinterpret_cast<uintx4*>(Cbuf + (b * COLS + r) * 128 + ((q ^ (r & 7)) * 16)) = v[i];
            }
        };
        uint32_t m1[2][2], m2[2][2];  // [row block][centroid block]
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                m1[a][b] = 0xFFFFFFFFu;
                m2[a][b] = 0xFFFFFFFFu;
            }
        floatx4 xa[XV], xb[XV];
        uintx4 cv[CV];
        for (int ct = 0; ct < ctiles; ++ct) {
            load_x(0, xa);
            load_c(ct, 0, cv);
            if (chunks > 1) load_x(1, xb);
            __syncthreads();  // the previous centroid tile's readers are done
            store_x(0, 0, xa, ct == 0);
            store_c(0, cv);
            __syncthreads();
            floatx16 acc[2][2];
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
            auto products = [&](int buf) {
                const unsigned char* xr = Xbuf + (buf * WIDE_ROWS + wr * 64 + r32) * 128;
                const unsigned char* cr = Cbuf + (buf * COLS + wc * 64 + r32) * 128;
                const int sw = r32 & 7;
                auto frag = [&](const unsigned char* p, int blk, int q) {
                    return __builtin_bit_cast(bf16x8,
                                              *reinterpret_cast<const uintx4*>(p + blk * 32 * 128 + ((q ^ sw) * 16)));
                };
                // small products first (km_assign_split.hpp): both steps' halves, then hi.hi
                bf16x8 xh[2][2], ch[2][2];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    bf16x8 xl[2], cl[2];
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        xh[s][a] = frag(xr, a, 2 * s + h);
                        xl[a] = frag(xr, a, 4 + 2 * s + h);
                        ch[s][a] = frag(cr, a, 2 * s + h);
                        cl[a] = frag(cr, a, 4 + 2 * s + h);
                    }
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int b = 0; b < 2; ++b) {
                            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ch[s][b], xl[a], acc[a][b], 0, 0, 0);
                            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cl[b], xh[s][a], acc[a][b], 0, 0, 0);
                        }
                }
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int b = 0; b < 2; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ch[s][b], xh[s][a], acc[a][b], 0, 0, 0);
            };
            // chunk c's products; chunk c + 1 goes to the other buffer behind them
            auto step = [&](int c, floatx4(&next)[XV], floatx4(&after)[XV]) {
                const bool more = c + 1 < chunks;
                if (more) load_c(ct, c + 1, cv);
                if (c + 2 < chunks) load_x(c + 2, after);
                products(c & 1);
                if (more) {
                    store_x(c + 1, (c + 1) & 1, next, ct == 0);
                    store_c((c + 1) & 1, cv);
                }
                __syncthreads();
            };
            int c = 0;
            for (; c + 1 < chunks; c += 2) {
                step(c, xb, xa);
                step(c + 1, xa, xb);
            }
            if (c < chunks) step(c, xb, xa);
            if (ct == 0) {
                // row norms: eight lanes of a row, chains of at most d / 8 additions
#pragma unroll
                for (int i = 0; i < XV; ++i) {
                    float t = sq[i];
                    t += __shfl_xor(t, 1);
                    t += __shfl_xor(t, 2);
                    t += __shfl_xor(t, 4);
                    const int r = (tid >> 3) + i * (T / 8);
                    if ((tid & 7) == 0) {
                        const float up = t * (1.0f + WIDE_NORM_UP);
                        // the last term: underflow of up to 4096 products (a split row's 2e-35 is for 128)
                        const float da = split_delta<3>(kc, up, C, 0.f, 0.f) + 1e-33f;
                        rx2[r] = t;
                        rda[r] = da;
                        rs_s[r] = (up + da) * (1.0f + 2.4e-7f);
                    }
                }
                __syncthreads();
            }
            // keys of this centroid tile
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int blk = (ct * COLS + wc * 64) / 32 + b;
                const uint32_t tag = uint32_t(blk) << 4;
                float cn[16];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const floatx4 c4 = *reinterpret_cast<const floatx4*>(cnw + blk * 32 + 8 * q + 4 * h);
#pragma unroll
                    for (int t = 0; t < 4; ++t) cn[4 * q + t] = c4[t];
                }
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    const float s = rs_s[wr * 64 + a * 32 + r32];
#pragma unroll
                    for (int i = 0; i < 16; i += 2) {
                        const uint32_t ka = (__float_as_uint((acc[a][b][i] + s) + cn[i]) & kmask) | (tag | i);
                        const uint32_t kb = (__float_as_uint((acc[a][b][i + 1] + s) + cn[i + 1]) & kmask) | (tag | (i + 1));
                        const uint32_t med = max(min(m1[a][b], ka), min(max(m1[a][b], ka), kb));
                        m2[a][b] = min(m2[a][b], med);
                        m1[a][b] = min(m1[a][b], min(ka, kb));
                    }
                }
            }
        }
        // every row's slots through LDS (the chunk buffers are free): slot (wc, b, h)
        uint2* slots = reinterpret_cast<uint2*>(smem_raw);  // [WIDE_ROWS][NSLOT + 1]
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
                slots[(wr * 64 + a * 32 + r32) * (NSLOT + 1) + (wc * 2 + b) * 2 + h] = make_uint2(m1[a][b], m2[a][b]);
        __syncthreads();
        int outcome = 0, cnt = 0;
        int64_t row = -1;
        uint32_t TK = 0;
        float T_ = 0.f, lo_add = 0.f;
        const uint2* mine = slots + (tid < WIDE_ROWS ? tid : 0) * (NSLOT + 1);
        auto idx_of = [&](uint32_t key, int sl) {
            const uint32_t low = key & ((1u << kc.ib) - 1u);
            const int i = int(low & 15u);
            return int(low >> 4) * 32 + 8 * (i >> 2) + 4 * (sl & 1) + (i & 3);
        };
        if (tid < WIDE_ROWS && rrow[tid] >= 0) {
            row = rrow[tid];
            uint32_t best = 0xFFFFFFFFu;
            int bs = 0;
            for (int q = 0; q < NSLOT; ++q)
                if (mine[q].x < best) {
                    best = mine[q].x;
                    bs = q;
                }
            const float X2 = rx2[tid], S = rs_s[tid], da = rda[tid];
            // as in assign_split_kernel
            const float v1 = __uint_as_float(best & kmask) * (1.0f + kc.trunc);
            const float d1 = fmaxf(0.f, ((v1 - S) + X2) + da + (WIDE_NORM_UP + 6e-7f) * (X2 + S) + 5e-7f * v1);
            T_ = (v1 + 2.0f * (da + kc.g_canon * d1)) * (1.0f + 6e-7f);
            lo_add = ((X2 - S) - da) - (WIDE_NORM_UP + 6e-7f) * (X2 + S);
            TK = (__float_as_uint(T_) & kmask) | ((1u << kc.ib) - 1u);
            bool cert = T_ < 1.0e38f && TK < 0x7F000000u;
            uint32_t second = 0xFFFFFFFFu;
            for (int q = 0; q < NSLOT; ++q) {
                const uint2 s = mine[q];
                cert = cert && s.y > TK;
                cnt += s.x <= TK ? 1 : 0;
                cert = cert && (s.x > TK || idx_of(s.x, q) < k);
                second = min(second, q == bs ? s.y : s.x);
            }
            if (cert && cnt == 1) {
                const int j = idx_of(best, bs);
                labels[row] = j;
                if (rs.gap)
                    rs.gap[row] = bound_gap(double(d1), double(__uint_as_float(second & kmask)) + double(lo_add), rs.gam,
                                            rs.base[j]);
            } else {
                outcome = cert && cnt <= MAXC ? 1 : 2;
            }
        }
        // one reservation per list and tile
        int at = 0;
        if (outcome) at = atomicAdd(&open_cnt[outcome - 1], 1);
        __syncthreads();
        if (tid < 2 && open_cnt[tid]) open_base[tid] = atomicAdd(&L.counters[tid], open_cnt[tid]);
        __syncthreads();
        if (outcome == 1) {
            const int e = open_base[0] + at;
            L.cand_rows[e] = int32_t(row);
            L.cand_count[e] = cnt;
            if (rs.gap) L.cand_lo[e] = float_below(double(T_) + double(lo_add));
            int c = 0;
            for (int q = 0; q < NSLOT; ++q)
                if (mine[q].x <= TK) L.cand_ids[int64_t(e) * MAXC + c++] = idx_of(mine[q].x, q);
        } else if (outcome == 2) {
            L.full_rows[open_base[1] + at] = int32_t(row);
        }
    }
}

}  // namespace km
