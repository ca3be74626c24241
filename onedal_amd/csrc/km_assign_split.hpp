// km_assign_split.hpp -- FP32 assignment on the BF16 matrix cores.
//
// float rows and centroids are split into two bf16 halves each, x = xh + xl + rx with
// |xl| <= 2^-9 |x| and |rx| <= 2^-18 |x|, and
//     2 x.c  ~  2 (xh.ch + xh.cl + xl.ch)
// is three v_mfma_f32_32x32x16_bf16 per 16 features, each 16 times the rate of
// v_mfma_f32_32x32x2f32: 5.3 times fewer matrix-core cycles than FP32 products.  The
// values only select candidates: like the FP32 and BF16 kernels (km_assign.hpp,
// km_assign_bf16.hpp) a row is settled when one centroid lies inside a proven
// error band and re-scored in the exact form otherwise, so the labels are those of
// the exact form whatever the products' precision.
//
// A lane tracks  v_j = ||c_j||^2 + s - 2 x.c_j,  s = ||x||^2 + its error bound (rounded
// up), so every v_j is positive and near the squared distance: the float bits order
// like the values, and a key (value bits, low IB bits replaced by block and
// register) loses only 2^(IB-23) of the distance itself.  s and ||c_j||^2 enter as one
// more matrix step (three exact bf16 pieces each against ones), so the accumulators
// start at zero and no row statistics are read: a row's norm is formed in the kernel.
//
// Error bound (X = ||x||, C = max ||c_j||):
//   split:        2 (|xl.cl| + |rx.c| + |x.rc|) <= 6.02 2^-18 X C
//   accumulation: gamma_m times the sum of the magnitudes so far (FP32, doubled unit
//                 roundoff, as in the other kernels).  The small products
//                 come first (their partial sums are below 2^-8 2 X C), then xh.ch,
//                 then the norms:
//                 gamma_2d 2.02 2^-8 X C + gamma_d 2.04 X C + gamma_8 1.02 (X + C)^2
//   rounding of ||c_j||^2, s: 2^-22 (X^2 + C^2); underflow of halves and products:
//                 1e-32 (X + C) + 2e-35
// Padding features are exact zeros and add nothing.
//
// TERMS = 1 keeps xh.ch alone: the BF16 form for rows that are assigned once
// (inference), straight from the float rows.  Its band is the BF16 one,
//   2 (X Ec + ex C (1 + 2^-8)) + gamma_d 2.04 X C + gamma_8 1.02 (X + C)^2 + ...
// with Ec = max ||c - bf16(c)|| and ex = ||x - bf16(x)|| formed in the kernel; rows that
// its slots cannot settle go through the three-term kernel, a list of rows.  A BF16
// copy of the rows would be written and read once for nothing: at n=5e6, d=128, k=512
// the conversion took 0.91 ms of a 1.57 ms call.  Training keeps the copy
// (assign_bf16_kernel): its passes read the rows again and again.
#pragma once

#include "km_assign.hpp"
#include "km_assign_bf16.hpp"
#include "km_bounds.hpp"
#include "km_common.hpp"

namespace km {

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// largest k of this path: its keys hold at most 11 index bits
constexpr int SPLIT_MAX_K = 4096;

// FP32 throughout: 1.03 in split_delta covers the rounding of the bound itself
struct split_consts {
    float xc;        // factor of X C
    float sum;       // factor of (X + C)^2
    float trunc;     // 2^(IB-23)
    float g_canon;   // g' of the exact-form distance
    int ib;
};

// value error of a row with squared norm at most X2 (one term: Ec, and ex2 = ex^2)
template <int TERMS>
__device__ __forceinline__ float split_delta(const split_consts& kc, float X2, float C, float Ec, float ex2) {
    const float X = sqrtf(X2), m = X + C;
    float e = kc.xc * X * C + kc.sum * m * m + 2.4e-7f * (X2 + C * C) + 1e-32f * m + 2e-35f;
    if (TERMS == 1) e += 2.0f * (X * Ec + sqrtf(ex2) * C * 1.004f);
    return 1.03f * e;
}

// (hi, lo) bf16 halves of two floats, packed
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    const bf2 h = __builtin_convertvector(f2{a, b}, bf2);
    hi = __builtin_bit_cast(uint32_t, h);
    const float ah = __uint_as_float(hi << 16), bh = __uint_as_float(hi & 0xFFFF0000u);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a - ah, b - bh}, bf2));
}

// three bf16 pieces whose sum is exactly v (v >= 0, finite): bits h | m << 16, l
__device__ __forceinline__ void split3(float v, uint32_t& hm, uint32_t& l) {
    const uint32_t h = __float_as_uint(v) & 0xFFFF0000u;
    const float r = v - __uint_as_float(h);
    const uint32_t m = __float_as_uint(r) & 0xFFFF0000u;
    const float r2 = r - __uint_as_float(m);
    hm = (h >> 16) | m;
    l = __float_as_uint(r2) >> 16;
}

// Ring of 4 LDS slots: a block of 32 centroids with both halves is 128 DP bytes, and
// 1 KB of norm pieces (DP = 128: 68 KB, two workgroups per CU)
constexpr int SPLIT_RING = 4;
__host__ inline size_t split_lds_bytes(int dp, int terms) {
    const size_t ring = size_t(SPLIT_RING) * (size_t(terms == 3 ? 128 : 64) * dp + 1024);
    return ring > 16384 ? ring : 16384;  // rows are transposed in it, 4 KB a wave
}

// Workgroup = 4 waves of NB x 32 rows (B operand, both halves in registers for the
// whole pass); blocks of 32 centroids (A operand) stream through the LDS ring by
// direct-to-LDS copies, one barrier per block, as in assign_bf16_kernel: 16-byte
// chunk c of a row sits at chunk c ^ (row & SWZ).  Lane l = 32 h + r holds row r's
// features 32 p + 16 h .. + 15 of every 128-byte piece p.  Rows are read as whole
// pieces (eight lanes a piece, so every load is full lines; a lane reading its own row
// 16 bytes at a time fetched each line from L2 again and again: 1.25 ms a launch at
// n=5e6, d=128, k=512) and pass through the ring's memory to their lanes before the
// ring is filled.  Cs: rows of [hi DP | lo DP] bf16 of -2 c_j, and
// cnp: 16 bf16 per row (the norm step's operand), both padded to whole groups of
// four blocks (padding: zero rows with a huge norm).  Slots and settling as in
// assign_bf16_kernel; rows without a certain candidate set go to the full list (one
// term: to the collect rows, for the three-term kernel).
template <int DP, int NB, int TERMS>
__global__ __launch_bounds__(256, 2) void assign_split_kernel(
    const float* __restrict__ X, int64_t n, int d, const uint16_t* __restrict__ Cs,
    const uint16_t* __restrict__ cnp, int k, const double* __restrict__ cmax_p, split_consts kc,
    int32_t* __restrict__ labels, refine_lists L, row_select rs) {
    constexpr int HALF = DP / 2;
    constexpr int STEPS = HALF / 8;
    constexpr int PIECES = DP / 32;  // 128-byte pieces of a row
    constexpr int ROWS_PER_WAVE = 32 * NB;
    constexpr int ROWS_PER_WG = 4 * ROWS_PER_WAVE;
    constexpr int ROWB = TERMS == 3 ? DP * 4 : DP * 2;  // bytes of a centroid row in LDS
    constexpr int CPR = ROWB / 16;                  // 16-byte chunks of it
    constexpr int SWZ = (CPR < 16 ? CPR : 16) - 1;  // chunk swizzle mask
    constexpr int BLKB = 32 * ROWB;
    constexpr int NDATA = BLKB / 1024;              // 1 KB copies per block
    constexpr int DPW = NDATA >= 4 ? NDATA / 4 : 1;  // of each wave (2 KB blocks: two waves copy the same)
    constexpr int CPW = DPW + 1;                    // + the block's norm pieces
    constexpr int NSL = 4;
    constexpr int RING = SPLIT_RING;
    constexpr int AHEAD = RING - 1;
    static_assert(DPW >= 1, "block copy layout");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int open_cnt[2][4], open_base[2];  // the tile's list entries per wave, and where they go
    unsigned char* ring = smem_raw;                          // [RING][BLKB]
    unsigned char* ring_cn = smem_raw + size_t(RING) * BLKB;  // [RING][1024]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int r32 = lane & 31;
    const int h = lane >> 5;
    const int mblocks = bf16_padded_k(k) / 32;  // a multiple of 4
    const float C = float(cmax_p[0]) * (1.0f + 2.4e-7f);
    const float Ec = TERMS == 1 ? float(cmax_p[2]) * (1.0f + 2.4e-7f) : 0.f;
    const uint32_t kmask = 0x7FFFFFFFu & ~((1u << kc.ib) - 1u);
    const int64_t nrows = select_rows(rs, n);
    const int64_t ntiles = (nrows + ROWS_PER_WG - 1) / ROWS_PER_WG;
    uint32_t kmv;
    asm volatile("v_mov_b32 %0, %1" : "=v"(kmv) : "s"(kmask));

    // this wave's copies of a block (see assign_bf16_kernel)
    uint32_t voff[DPW], moff[DPW];
#pragma unroll
    for (int c = 0; c < DPW; ++c) {
        const int q = NDATA >= 4 ? wave + 4 * c : wave % NDATA;
        const int p = q * 64 + lane;
        const int prow = p / CPR, pc = p % CPR;
        voff[c] = uint32_t(prow * DP * 4 + (pc ^ (prow & SWZ)) * 16);  // both halves in memory
        moff[c] = lds_addr(ring + q * 1024);
    }
    const uint32_t voff_cn = uint32_t(lane * 16);
    const uint32_t moff_cn = lds_addr(ring_cn);
    auto issue_block = [&](int mb, int slot) {
        const void* gb = uniform_ptr(reinterpret_cast<const unsigned char*>(Cs) + size_t(mb) * (128 * DP));
#pragma unroll
        for (int c = 0; c < DPW; ++c) lds_dma16(gb, voff[c], moff[c] + slot * BLKB);
        const void* gc = uniform_ptr(reinterpret_cast<const unsigned char*>(cnp) + size_t(mb) * 1024);
        lds_dma16(gc, voff_cn, moff_cn + slot * 1024);
    };

    // rows of a tile: loaded as floats while the previous tile settles, then split into
    // both halves, the norm step's operand, and what the settle needs
    uintx4 xh[NB][STEPS], xl[NB][TERMS == 3 ? STEPS : 1];
    uintx4 xs_op[NB];
    floatx4 raw[NB][PIECES][4];
    int64_t rows[NB];
    float x2[NB], xs[NB], da[NB];
    auto load_tile = [&](int64_t tile) {
        const int64_t w0 = tile * ROWS_PER_WG + int64_t(wave) * ROWS_PER_WAVE;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int64_t own = w0 + nb * 32 + r32;
            rows[nb] = own < nrows ? select_row(rs, own) : -1;
            // this lane's 16 bytes of rows lane / 8 + 8 i
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t e = w0 + nb * 32 + 8 * i + (lane >> 3);
                const bool ok = e < nrows;
                const int64_t row = ok ? select_row(rs, e) : 0;
                const float* src = X + row * d + 4 * (lane & 7);
                // 16-byte loads need dword alignment only, so any width takes them.  The
                // last vector of an odd width also reads the next row's first features
                // (masked in split_tile); the last row of X has none: by elements.
                const int left = ok ? d - 4 * (lane & 7) : 0;               // features from src on
                const int64_t avail = (n - row) * d - 4 * (lane & 7);  // floats from src to the end of X
#pragma unroll
                for (int p = 0; p < PIECES; ++p) {
                    floatx4 t = {0.f, 0.f, 0.f, 0.f};
                    if (32 * p < left) {
                        if (32 * p + 4 <= avail) {
                            t = *reinterpret_cast<const floatx4u*>(src + 32 * p);
                        } else {
                            t[0] = src[32 * p];
                            if (32 * p + 1 < left) t[1] = src[32 * p + 1];
                            if (32 * p + 2 < left) t[2] = src[32 * p + 2];
                        }
                    }
                    raw[nb][p][i] = t;
                }
            }
        }
    };
    // each row's pieces to the lanes that hold it (the ring is empty; a wave uses 4 KB of
    // it, and its LDS operations run in order)
    auto transpose_tile = [&]() {
        unsigned char* mine = ring + wave * 4096;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int p = 0; p < PIECES; ++p) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = 8 * i + (lane >> 3);
                    *reinterpret_cast<floatx4*>(mine + r * 128 + (((lane & 7) ^ (r & 7)) * 16)) = raw[nb][p][i];
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    raw[nb][p][q] =
                        *reinterpret_cast<const floatx4*>(mine + r32 * 128 + (((4 * h + q) ^ (r32 & 7)) * 16));
                __builtin_amdgcn_wave_barrier();
            }
    };
    auto split_tile = [&]() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            float sq[4] = {0.f, 0.f, 0.f, 0.f}, se[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 2 * STEPS; ++q) {  // vector q: features 32 (q / 4) + 16 h + 4 (q % 4) ..
                floatx4 v = raw[nb][q >> 2][q & 3];
                if (d & 3) {
                    const int left = d - 32 * (q >> 2) - 16 * h - 4 * (q & 3);
#pragma unroll
                    for (int u = 1; u < 4; ++u) v[u] = u < left ? v[u] : 0.f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) sq[u] = __builtin_fmaf(v[u], v[u], sq[u]);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    uint32_t hi, lo;
                    split2(v[2 * u], v[2 * u + 1], hi, lo);  // one term: lo is not used
                    xh[nb][q >> 1][2 * (q & 1) + u] = hi;
                    if constexpr (TERMS == 3) {
                        xl[nb][q >> 1][2 * (q & 1) + u] = lo;
                    } else {
                        const float e0 = v[2 * u] - __uint_as_float(hi << 16);
                        const float e1 = v[2 * u + 1] - __uint_as_float(hi & 0xFFFF0000u);
                        se[2 * u] = __builtin_fmaf(e0, e0, se[2 * u]);
                        se[2 * u + 1] = __builtin_fmaf(e1, e1, se[2 * u + 1]);
                    }
                }
            }
            // ||x||^2: chains of at most DP / 8 additions, so the relative error is
            // below (DP / 8 + 4) 2^-24
            float t = (sq[0] + sq[1]) + (sq[2] + sq[3]);
            t += __shfl_xor(t, 32);
            x2[nb] = t;
            const float up = t * (1.0f + 2.4e-6f);
            float ex2 = 0.f;
            if constexpr (TERMS == 1) {
                ex2 = (se[0] + se[1]) + (se[2] + se[3]);
                ex2 = (ex2 + __shfl_xor(ex2, 32)) * (1.0f + 2.4e-6f);
            }
            da[nb] = split_delta<TERMS>(kc, up, C, Ec, ex2);
            xs[nb] = (up + da[nb]) * (1.0f + 2.4e-7f);
            uint32_t hm, l;
            split3(xs[nb], hm, l);
            // slots: [1 1 1 s_h s_m s_l 0 0] against [c_h c_m c_l 1 1 1 0 0]
            const uintx4 op = {0x3F803F80u, 0x00003F80u | (hm << 16), (hm >> 16) | (l << 16), 0u};
            xs_op[nb] = h == 0 ? op : uintx4{0u, 0u, 0u, 0u};
        }
    };
    load_tile(blockIdx.x);
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        uint32_t m1[NB][NSL], m2[NB][NSL];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int q = 0; q < NSL; ++q) {
                m1[nb][q] = 0xFFFFFFFFu;
                m2[nb][q] = 0xFFFFFFFFu;
            }
        auto mfma_block = [&](int slot, floatx16(&acc)[NB]) {
            const unsigned char* arow = ring + slot * BLKB + r32 * ROWB;
            const bf16x8 an = __builtin_bit_cast(
                bf16x8, *reinterpret_cast<const uintx4*>(ring_cn + slot * 1024 + r32 * 32 + h * 16));
            bf16x8 ah[STEPS], al[TERMS == 3 ? STEPS : 1];
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int c = 4 * (s >> 1) + 2 * h + (s & 1);  // step s: features 8 c .. 8 c + 7
                ah[s] = __builtin_bit_cast(
                    bf16x8, *reinterpret_cast<const uintx4*>(arow + ((c ^ (r32 & SWZ)) * 16)));
                if constexpr (TERMS == 3)
                    al[s] = __builtin_bit_cast(
                        bf16x8, *reinterpret_cast<const uintx4*>(arow + (((DP / 8 + c) ^ (r32 & SWZ)) * 16)));
            }
            // the small products first, then xh.ch, then the norms (the error bound
            // counts on this order)
            const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if constexpr (TERMS == 3) {
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            ah[s], __builtin_bit_cast(bf16x8, xl[nb][s]), s == 0 ? zero : acc[nb], 0, 0, 0);
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            al[s], __builtin_bit_cast(bf16x8, xh[nb][s]), acc[nb], 0, 0, 0);
                }
            }
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        ah[s], __builtin_bit_cast(bf16x8, xh[nb][s]), TERMS == 1 && s == 0 ? zero : acc[nb], 0, 0, 0);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(an, __builtin_bit_cast(bf16x8, xs_op[nb]), acc[nb],
                                                                  0, 0, 0);
        };
        // keys of block mb into slot sl (running top-2), as in assign_bf16_kernel
        auto keys_block = [&](const floatx16(&acc)[NB], int mb, int sl) {
            const uint32_t tag = uint32_t(mb) << 4;
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                uint32_t ta, tb;
                asm("s_or_b32 %0, %1, %2" : "=s"(ta) : "s"(tag), "i"(i) : "scc");
                asm("s_or_b32 %0, %1, %2" : "=s"(tb) : "s"(tag), "i"(i + 1) : "scc");
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const uint32_t ka = (__float_as_uint(acc[nb][i]) & kmv) | ta;
                    const uint32_t kb = (__float_as_uint(acc[nb][i + 1]) & kmv) | tb;
                    const uint32_t med = max(min(m1[nb][sl], ka), min(max(m1[nb][sl], ka), kb));
                    m2[nb][sl] = min(m2[nb][sl], med);
                    m1[nb][sl] = min(m1[nb][sl], min(ka, kb));
                }
            }
        };
        floatx16 acc0[NB], acc1[NB];
        auto step = [&](int mb, int u, floatx16(&cur)[NB], floatx16(&prev)[NB]) {
            // nothing is scheduled across the wait, the barrier and the copies
            __builtin_amdgcn_sched_barrier(0);
            wait_vm<(AHEAD - 1) * CPW>();
            __syncthreads();
            issue_block(min(mb + AHEAD, mblocks - 1), (mb + AHEAD) & (RING - 1));
            __builtin_amdgcn_sched_barrier(0);
            mfma_block(mb & (RING - 1), cur);
            keys_block(prev, mb - 1, (u + 3) & 3);
        };
        // row loads complete here; the previous tile's last readers are done before
        // the prologue refills the ring
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __syncthreads();
        transpose_tile();
        __syncthreads();
#pragma unroll
        for (int b = 0; b < AHEAD; ++b) issue_block(min(b, mblocks - 1), b);
        split_tile();  // while the first blocks are on their way
        __builtin_amdgcn_sched_barrier(0);
        // the first step's "previous block": keys above every real one
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc1[nb][i] = __uint_as_float(0xFFFFFFFFu);
        for (int mb = 0; mb < mblocks; mb += 4) {
            step(mb, 0, acc0, acc1);
            step(mb + 1, 1, acc1, acc0);
            step(mb + 2, 2, acc0, acc1);
            step(mb + 3, 3, acc1, acc0);
        }
        keys_block(acc1, mblocks - 1, 3);
        // the next tile's rows load while this tile settles, in the registers of the
        // accumulators (hence the barriers: no load moves up among the last keys, no
        // split down into the block loop)
        __builtin_amdgcn_sched_barrier(0);
        int64_t rows_s[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) rows_s[nb] = rows[nb];
        load_tile(tile + gridDim.x);  // past the last tile: no row, nothing read

        // settle: with two row blocks, lane (r32, h) settles row r32 of block h; with one
        // the lanes h = 0 settle
        const int nbs = NB == 2 ? h : 0;
        uint32_t k1[2 * NSL], k2[2 * NSL];  // own half's slots, then the partner's
#pragma unroll
        for (int q = 0; q < NSL; ++q) {
            k1[q] = nbs ? m1[NB - 1][q] : m1[0][q];
            k2[q] = nbs ? m2[NB - 1][q] : m2[0][q];
            const uint32_t s1 = (NB == 2 && !h) ? m1[NB - 1][q] : m1[0][q];
            const uint32_t s2 = (NB == 2 && !h) ? m2[NB - 1][q] : m2[0][q];
            k1[NSL + q] = __shfl_xor(s1, 32);
            k2[NSL + q] = __shfl_xor(s2, 32);
        }
        const int64_t row = nbs ? rows_s[NB - 1] : rows_s[0];
        const float X2 = nbs ? x2[NB - 1] : x2[0];
        const float S = nbs ? xs[NB - 1] : xs[0];
        const float dv = nbs ? da[NB - 1] : da[0];
        const bool active = (NB == 2 || h == 0) && row >= 0;
        auto idx_of = [&](uint32_t key, int hh) {
            const uint32_t low = key & ((1u << kc.ib) - 1u);
            const int mbk = int(low >> 4), i = int(low & 15u);
            return mbk * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);
        };
        uint32_t bo = k1[0], bp = k1[NSL];
#pragma unroll
        for (int q = 1; q < NSL; ++q) {
            bo = min(bo, k1[q]);
            bp = min(bp, k1[NSL + q]);
        }
        const uint32_t best = min(bo, bp);
        const int hb = bo <= bp ? h : 1 - h;
        // the best centroid's value lies in [v, v (1 + trunc)); its squared distance is
        // at most d1.  FP32: the last terms cover these sums' own rounding.
        const float v1 = __uint_as_float(best & kmask) * (1.0f + kc.trunc);
        const float d1 = fmaxf(0.f, ((v1 - S) + X2) + dv + 3e-6f * (X2 + S) + 5e-7f * v1);
        const float T = (v1 + 2.0f * (dv + kc.g_canon * d1)) * (1.0f + 6e-7f);
        // value -> lower bound of the squared distance
        const float lo_add = ((X2 - S) - dv) - 3e-6f * (X2 + S);
        // value(key) <= T  <=>  key <= TK (see assign_bf16_kernel); a threshold as high as
        // the padding's values, or one that is not a number, certifies nothing
        const uint32_t TK = (__float_as_uint(T) & kmask) | ((1u << kc.ib) - 1u);
        bool cert = T < 1.0e38f && TK < 0x7F000000u;
        int cnt = 0;
#pragma unroll
        for (int q = 0; q < 2 * NSL; ++q) {
            cert = cert && k2[q] > TK;
            cnt += k1[q] <= TK ? 1 : 0;
            cert = cert && (k1[q] > TK || idx_of(k1[q], q < NSL ? h : 1 - h) < k);
        }
        int outcome = 0;  // 1: candidate entry, 2: full entry
        if (active) {
            if (cert && cnt == 1) {
                const int j = idx_of(best, hb);
                labels[row] = j;
                if (rs.gap) {
                    uint32_t second = 0xFFFFFFFFu;
#pragma unroll
                    for (int q = 0; q < 2 * NSL; ++q) {
                        const bool own = k1[q] == best && (q < NSL ? h : 1 - h) == hb;
                        second = min(second, own ? k2[q] : k1[q]);
                    }
                    rs.gap[row] = bound_gap(double(d1), double(__uint_as_float(second & kmask)) + double(lo_add), rs.gam,
                                            rs.base[j]);
                }
            } else {
                outcome = cert ? 1 : 2;
            }
        }
        const uint64_t mc = __ballot(outcome == 1);
        const uint64_t ml = __ballot(outcome == 2);
        // one reservation per list and tile: every wave's atomics on the two counters
        // were the time of a pass over few rows (1M open rows of n=1e7: 0.39 ms)
        if (lane == 0) {
            open_cnt[0][wave] = int(__popcll(mc));
            open_cnt[1][wave] = int(__popcll(ml));
        }
        __syncthreads();
        const int tc = open_cnt[0][0] + open_cnt[0][1] + open_cnt[0][2] + open_cnt[0][3];
        const int tl = open_cnt[1][0] + open_cnt[1][1] + open_cnt[1][2] + open_cnt[1][3];
        if (tc + tl == 0) continue;  // uniform over the workgroup
        if (tid < 2) open_base[tid] = atomicAdd(&L.counters[tid == 0 ? 0 : TERMS == 3 ? 1 : 2], tid == 0 ? tc : tl);
        __syncthreads();
        int e0 = open_base[0], f0 = open_base[1];
        for (int w = 0; w < wave; ++w) {
            e0 += open_cnt[0][w];
            f0 += open_cnt[1][w];
        }
        if (mc) {
            if (outcome == 1) {
                const int e = e0 + lanes_below(mc);
                L.cand_rows[e] = int32_t(row);
                L.cand_count[e] = cnt;
                if (rs.gap) L.cand_lo[e] = float_below(double(T) + double(lo_add));
                int c = 0;
#pragma unroll
                for (int q = 0; q < 2 * NSL; ++q)
                    if (k1[q] <= TK) L.cand_ids[int64_t(e) * MAXC + c++] = idx_of(k1[q], q < NSL ? h : 1 - h);
            }
        }
        if (outcome == 2) (TERMS == 3 ? L.full_rows : L.coll_rows)[f0 + lanes_below(ml)] = int32_t(row);
    }
}

}  // namespace km
