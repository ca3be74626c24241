// km_assign_wide.hpp -- FP32 assignment of wide rows (d > 128) on the BF16 matrix cores.
//
// The split products and the settling of km_assign_split.hpp, for rows whose pieces do
// not fit a wave's registers: a tiled product over chunks of 32 features.  It replaces
// a VALU tile kernel for d > 256 (inference of n=1e5, d=512, k=256: 978 -> 307 us) and the
// FP32 matrix-core kernel for 128 < d <= 256 (n=1e6, d=200, k=300: 2.26 -> 1.39 ms).
//
// Workgroup = 8 waves, NWR x NWC, on a tile of 64 NWR rows x 64 NWC centroids; a wave owns
// 64 x 64 (two row blocks, two centroid blocks).  Per chunk a row is one full 128-byte
// line of X, read by eight lanes, split into its three bf16 pieces once and staged in
// LDS; the centroids' pieces, laid out chunk by chunk by the centroid step, so that a
// tile's chunk is one contiguous run, are copied there directly.  The first two
// pieces of a row are 128 bytes, 16-byte vector q of row r at q ^ (r & 7); the third
// pieces of two rows share a line, swizzled by line.  Two buffers; the next chunk's
// loads are in flight during the products.  2 x 4 waves read the rows once for k <= 256;
// 4 x 2, for k <= 128, leave no wave on padding.  One workgroup per CU (147 KB of LDS).
// Bound: per chunk a wave's 48 products take 1536 cycles and its LDS reads 24 KB, a half of
// that time at two waves per SIMD; n=1e5, d=512, k=256 takes 0.20 ms for all rows.
//
// The small products have accumulators of their own (64 more registers a lane), which join
// the others at the end: added to the large sums chunk by chunk, each would be bounded
// against all of 2 X C, and the band would be six times as wide.  Error bound: as
// in km_assign_split.hpp, but the norm and the small sums are added in FP32 after the
// products.
//
// Every lane keeps a top-2 slot per (row block, centroid block); a row's 4 NWC slots meet in
// LDS after the last centroid tile and one thread settles the row.
#pragma once

#include "km_assign_split.hpp"

namespace km {

__host__ __device__ constexpr int wide_rows(int nwc) { return 64 * (8 / nwc); }
__host__ __device__ constexpr int wide_cols(int nwc) { return 64 * nwc; }
// rows of the centroid operand, kp x whole chunks of 32 features x three pieces
__host__ inline int wide_kp(int k, int nwc) { return (k + wide_cols(nwc) - 1) / wide_cols(nwc) * wide_cols(nwc); }
__host__ __device__ inline int wide_chunks(int d) { return (d + 31) / 32; }
constexpr int WIDE_ROW = 32 * SPLIT_PIECES;  // bf16 of a row's chunk
__host__ inline size_t wide_lds_bytes(int nwc) {
    return size_t(2) * 2 * WIDE_ROW * (wide_cols(nwc) + wide_rows(nwc));
}

// Cw: [chunk][kp][c1 32 | c2 32 | c3 32] bf16 of -2 c; cnw: kp values ||c_j||^2 (padding: huge)
template <int NWC>
__global__ __launch_bounds__(512, 2) void assign_wide_kernel(
    const float* __restrict__ X, int64_t n, int d, const uint16_t* __restrict__ Cw, const float* __restrict__ cnw,
    int k, int kp, const double* __restrict__ cmax_p, split_consts kc, int32_t* __restrict__ labels,
    refine_lists L, row_select rs) {
    constexpr int T = 512;                  // threads
    constexpr int ROWS = wide_rows(NWC), COLS = wide_cols(NWC);
    constexpr int XV = ROWS * 8 / T;        // 16-byte vectors of X per thread and chunk
    constexpr int NSLOT = 4 * NWC;          // slots of a row: NWC waves x 2 blocks x 2 halves
    static_assert(COLS % 128 == 0 && ROWS <= T, "whole copies per wave, a thread per row");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    // [2 buffers] of [rows][128] for the first two pieces, then [rows / 2][128] for the third
    constexpr int CB = COLS * WIDE_ROW * 2, XB = ROWS * WIDE_ROW * 2;
    unsigned char* Cbuf = smem_raw;
    unsigned char* Xbuf = smem_raw + 2 * CB;
    __shared__ double rx[ROWS];  // ||x|| rounded up
    __shared__ int32_t rrow[ROWS];
    __shared__ int open_cnt[2], open_base[2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / NWC, wc = wave % NWC;  // row and column part of the wave
    const int r32 = lane & 31, h = lane >> 5;
    const int chunks = wide_chunks(d);
    const int ctiles = kp / COLS;
    const int64_t nsel = select_rows(rs, n);
    const int64_t ntiles = (nsel + ROWS - 1) / ROWS;
    // byte of 16-byte vector q of row r's piece in a buffer of `count` rows
    auto at = [](int count, int r, int piece, int q) {
        return piece < 2 ? r * 128 + (((4 * piece + q) ^ (r & 7)) * 16)
                         : count * 128 + (r >> 1) * 128 + (((4 * (r & 1) + q) ^ ((r >> 1) & 7)) * 16);
    };
    // this wave's copies of a centroid chunk: 1 KB, eight lines of a buffer each, of the first
    // two pieces (COLS lines) and of the third (COLS / 2)
    const int cline = wave * 8 + (lane >> 3), cvec = (lane & 7) ^ (cline & 7);
    const uint32_t voff12 = uint32_t(cline * (WIDE_ROW * 2) + cvec * 16);
    const uint32_t voff3 = uint32_t((2 * cline + (cvec >> 2)) * (WIDE_ROW * 2) + 128 + (cvec & 3) * 16);
    const uint32_t moff = lds_addr(Cbuf + wave * 1024);
    auto copy_c = [&](int ct, int c, int b) {
        const unsigned char* src =
            reinterpret_cast<const unsigned char*>(Cw + (int64_t(c) * kp + int64_t(ct) * COLS) * WIDE_ROW);
#pragma unroll
        for (int i = 0; i < COLS / 64; ++i)
            lds_dma16(uniform_ptr(src + i * 64 * (WIDE_ROW * 2)), voff12, moff + b * CB + i * 8192);
#pragma unroll
        for (int i = 0; i < COLS / 128; ++i)
            lds_dma16(uniform_ptr(src + i * 128 * (WIDE_ROW * 2)), voff3, moff + b * CB + COLS * 128 + i * 8192);
    };
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t n0 = tile * ROWS;
        __syncthreads();  // the previous tile's readers are done
        if (tid < ROWS) rrow[tid] = n0 + tid < nsel ? int32_t(select_row(rs, n0 + tid)) : -1;
        if (tid < 2) open_cnt[tid] = 0;
        __syncthreads();
        // this thread's vectors: row tid / 8 + i T / 8, vector tid % 8 of each chunk
        int xrow[XV];
#pragma unroll
        for (int i = 0; i < XV; ++i) xrow[i] = rrow[(tid >> 3) + i * (T / 8)];
        const int xleft = d - 4 * (tid & 7);  // features from this thread's vector on
        auto load_x = [&](int c, floatx4(&v)[XV]) {
            const int f = 32 * c;
#pragma unroll
            for (int i = 0; i < XV; ++i) {
                floatx4 t = {0.f, 0.f, 0.f, 0.f};
                if (f < xleft && xrow[i] >= 0) {
                    const float* src = X + int64_t(xrow[i]) * d + 4 * (tid & 7) + f;
                    if (f + 4 <= xleft || xrow[i] + 1 < n) {  // past the row only where rows follow
                        t = *reinterpret_cast<const floatx4u*>(src);
                    } else {
                        t[0] = src[0];
                        if (f + 1 < xleft) t[1] = src[1];
                        if (f + 2 < xleft) t[2] = src[2];
                    }
                }
                v[i] = t;
            }
        };
        double sq[XV];
#pragma unroll
        for (int i = 0; i < XV; ++i) sq[i] = 0.0;
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
                    for (int u = 0; u < 4; ++u) sq[i] = fma(double(x[u]), double(x[u]), sq[i]);
                }
                uint32_t a[3], e[3];
                split_pair(x[0], x[1], a[0], a[1], a[2]);
                split_pair(x[2], x[3], e[0], e[1], e[2]);
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    *reinterpret_cast<uint2*>(Xbuf + b * XB + at(ROWS, r, p, q >> 1) + (q & 1) * 8) =
                        make_uint2(a[p], e[p]);
            }
        };
        split_slot st[2][2];  // [row block][centroid block]
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) st[a][b].init();
        floatx4 xv[XV];
        for (int ct = 0; ct < ctiles; ++ct) {
            load_x(0, xv);
            __syncthreads();  // the previous centroid tile's readers are done
            copy_c(ct, 0, 0);
            store_x(0, 0, xv, ct == 0);
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's copies have arrived
            __syncthreads();
            floatx16 acc[2][2], low[2][2];
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        acc[a][b][i] = 0.f;
                        low[a][b][i] = 0.f;
                    }
            auto products = [&](int buf) {
                auto xfrag = [&](int blk, int piece, int s) {
                    return __builtin_bit_cast(
                        bf16x8, *reinterpret_cast<const uintx4*>(
                                    Xbuf + buf * XB + at(ROWS, wr * 64 + blk * 32 + r32, piece, 2 * s + h)));
                };
                auto cfrag = [&](int blk, int piece, int s) {
                    return __builtin_bit_cast(
                        bf16x8, *reinterpret_cast<const uintx4*>(
                                    Cbuf + buf * CB + at(COLS, wc * 64 + blk * 32 + r32, piece, 2 * s + h)));
                };
                auto mac = [&](floatx16(&to)[2][2], const bf16x8(&c)[2], const bf16x8(&x)[2]) {
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int b = 0; b < 2; ++b)
                            to[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[b], x[a], to[a][b], 0, 0, 0);
                };
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    bf16x8 x1[2], x2[2], x3[2], c1[2], c2[2], c3[2];
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        x1[a] = xfrag(a, 0, s);
                        x2[a] = xfrag(a, 1, s);
                        x3[a] = xfrag(a, 2, s);
                        c1[a] = cfrag(a, 0, s);
                        c2[a] = cfrag(a, 1, s);
                        c3[a] = cfrag(a, 2, s);
                    }
                    mac(low, c1, x3);
                    mac(low, c3, x1);
                    mac(low, c2, x2);
                    mac(low, c1, x2);
                    mac(low, c2, x1);
                    mac(acc, c1, x1);
                }
            };
            // chunk c's products; chunk c + 1 goes to the other buffer beside them
            for (int c = 0; c < chunks; ++c) {
                const bool more = c + 1 < chunks;
                if (more) {
                    copy_c(ct, c + 1, (c + 1) & 1);
                    load_x(c + 1, xv);
                }
                products(c & 1);
                if (more) store_x(c + 1, (c + 1) & 1, xv, ct == 0);
                __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), as above
                __syncthreads();
            }
            // values of this centroid tile
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int blk = (ct * COLS + wc * 64) / 32 + b;
                float cn[16];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const floatx4 c4 = *reinterpret_cast<const floatx4*>(cnw + blk * 32 + 8 * q + 4 * h);
#pragma unroll
                    for (int t = 0; t < 4; ++t) cn[4 * q + t] = c4[t];
                }
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    const float was = st[a][b].m1;
#pragma unroll
                    for (int i = 0; i < 16; ++i) st[a][b].push((acc[a][b][i] + low[a][b][i]) + cn[i], i);
                    st[a][b].id = st[a][b].m1 < was ? st[a][b].id | (blk << 4) : st[a][b].id;
                }
            }
        }
        // row norms: eight lanes of a row
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            double t = sq[i];
            t += __shfl_xor(t, 1);
            t += __shfl_xor(t, 2);
            t += __shfl_xor(t, 4);
            if ((tid & 7) == 0) rx[(tid >> 3) + i * (T / 8)] = sqrt(t) * (1.0 + 1e-12);
        }
        // every row's slots through LDS (the chunk buffers are free): slot (wc, b, h)
        split_slot* slots = reinterpret_cast<split_slot*>(smem_raw);  // [ROWS][NSLOT + 1]
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
                slots[(wr * 64 + a * 32 + r32) * (NSLOT + 1) + (wc * 2 + b) * 2 + h] = st[a][b];
        __syncthreads();
        int outcome = 0, cnt = 0;
        int64_t row = -1;
        float TF = 0.f;
        double other = 0.0;
        const split_slot* mine = slots + (tid < ROWS ? tid : 0) * (NSLOT + 1);
        auto idx_of = [&](int id, int sl) {
            const int i = id & 15;
            return (id >> 4) * 32 + 8 * (i >> 2) + 4 * (sl & 1) + (i & 3);
        };
        if (tid < ROWS && rrow[tid] >= 0) {
            row = rrow[tid];
            float best = mine[0].m1;
            int bs = 0;
            for (int q = 1; q < NSLOT; ++q)
                if (mine[q].m1 < best) {
                    best = mine[q].m1;
                    bs = q;
                }
            // as in assign_split_kernel
            const split_band b = make_split_band(kc, rx[tid], *cmax_p, best);
            TF = b.TF;
            other = split_lo(b, b.T);
            bool cert = b.in_range;
            float second = __builtin_inff();
            for (int q = 0; q < NSLOT; ++q) {
                const split_slot s = mine[q];
                const bool cand = s.m1 <= TF;
                cert = cert && s.m2 > TF && (!cand || idx_of(s.id, q) < k);
                cnt += cand ? 1 : 0;
                const float v = q == bs ? s.m2 : s.m1;
                second = v < second ? v : second;
            }
            if (cert && cnt == 1) {
                const int j = idx_of(mine[bs].id, bs);
                labels[row] = j;
                if (rs.gap)
                    rs.gap[row] = bound_gap(split_up(b, best), split_lo(b, double(second)), rs.gam, rs.base[j]);
            } else {
                outcome = cert && cnt > 0 && cnt <= MAXC ? 1 : 2;
            }
        }
        // one reservation per list and tile
        int pos = 0;
        if (outcome) pos = atomicAdd(&open_cnt[outcome - 1], 1);
        __syncthreads();
        if (tid < 2 && open_cnt[tid]) open_base[tid] = atomicAdd(&L.counters[tid], open_cnt[tid]);
        __syncthreads();
        if (outcome == 1) {
            const int e = open_base[0] + pos;
            L.cand_rows[e] = int32_t(row);
            L.cand_count[e] = cnt;
            if (rs.gap) L.cand_lo[e] = float_below(other);
            int c = 0;
            for (int q = 0; q < NSLOT; ++q)
                if (mine[q].m1 <= TF) L.cand_ids[int64_t(e) * MAXC + c++] = idx_of(mine[q].id, q);
        } else if (outcome == 2) {
            L.full_rows[open_base[1] + pos] = int32_t(row);
        }
    }
}

}  // namespace km
