// km_assign_split.hpp -- FP32 assignment on the BF16 matrix cores.
//
// A float is the sum of three bf16 pieces, x = x1 + x2 + x3 with |x2| <= 2^-9 |x| and
// |x3| <= 2^-18 |x|, and
//     2 x.c  =  2 (x1.c1 + x2.c1 + x1.c2 + x2.c2 + x3.c1 + x1.c3)
// up to 2^-25 X C (X = ||x||, C = max ||c_j||), less than one FP32 rounding per product: six
// v_mfma_f32_32x32x16_bf16 per 16 features, each 16 times the rate of
// v_mfma_f32_32x32x2f32, so 2.7 times fewer matrix-core cycles than FP32 products.  The
// products are no less accurate than FP32 ones: against 64 bits, over mixtures of d = 4
// to 4096 columns, near the origin, anisotropic and far from it, the root mean square
// error of ||c||^2 - 2 x.c is 0.07-0.93 of the FP32 matrix cores', the largest error
// 0.03-0.85 of theirs (d > 128: in km_assign_wide.hpp's order).  Two pieces and three
// products had up to 85 times their error at d = 4 and 17 at d = 128.  At d = 1 and 2, one
// or two products a value, FP32 products err less (0.6-0.9 of these), d = 3 is even: narrower
// rows than four columns take FP32 products.  Inference calls on (n, d, k), FP32 products and
// these: (1e6, 4, 256) 426 and 155 us, (1e6, 64, 256) 589 and 257, (2e5, 128, 4096) 3087 and
// 1250; three products took 130, 184 and 815.
//
// As in the other kernels (km_assign.hpp, km_assign_bf16.hpp) a row is settled when one
// centroid lies inside a proven error band and re-scored in the exact form otherwise,
// so the labels are those of the exact form.  A lane tracks v_j = ||c_j||^2 - 2 x.c_j in
// FP32, a top-2 per slot with the first one's index, and settles in double.
// ||c_j||^2 enters as one more matrix step: three exact bf16 pieces against ones.
//
// Error bound of v_j (FP32 accumulation: gamma_m, doubled unit roundoff, of the
// magnitudes so far, as in the other kernels).  The five small products come first:
// their partial sums stay below (2 + 0.03) 2^-8 X C; then x1.c1, then the norm:
//     left out:      1.05 2^-25 X C
//     accumulation:  gamma_5d 2.03 2^-8 X C + gamma_d 2.02 X C + gamma_4 (2.05 X C + 1.01 C^2)
//     ||c_j||^2:     1.01 2^-24 C^2 + gamma_d (2^-52) C^2
//     underflow of pieces and products: 1e-32 (X + C) + 2e-35
// Padding features are exact zeros and add nothing.  Norms whose products could pass
// the float range settle nothing.
//
// PIECES = 1 keeps x1.c1 alone: the BF16 form for rows that are assigned once
// (inference), straight from the float rows.  Its lanes track
// v_j = ||c_j||^2 + s - 2 x.c_j,  s = ||x||^2 + its error bound (rounded up), so every v_j is
// positive and near the squared distance: the float bits order like the values, and a
// key (value bits, low IB bits replaced by block and register) loses only 2^(IB-23) of the
// distance itself.  s enters in the norm step.  Its band is the BF16 one,
//   2 (X Ec + ex C (1 + 2^-8)) + gamma_d 2.04 X C + gamma_8 1.02 (X + C)^2 + ...
// with Ec = max ||c - bf16(c)|| and ex = ||x - bf16(x)|| formed in the kernel; rows that
// its slots cannot settle go through the three-piece kernel, a list of rows.  A BF16
// copy of the rows would be written and read once for nothing: at n=5e6, d=128, k=512
// the conversion took 0.91 ms of a 1.57 ms call.  Training keeps the copy
// (assign_bf16_kernel): its passes read the rows again and again.
#pragma once

#include <type_traits>

#include "km_assign.hpp"
#include "km_assign_bf16.hpp"
#include "km_bounds.hpp"
#include "km_common.hpp"

namespace km {

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// largest k of this path: the one-piece keys hold at most 11 index bits, and the centroids'
// pieces (3 MB at d = 128) stay in an XCD's L2; the other side was not measured
constexpr int SPLIT_MAX_K = 4096;
// narrowest rows whose products have no larger error than FP32 ones (see above)
constexpr int SPLIT_MIN_D = 4;
// bf16 pieces of a centroid feature
constexpr int SPLIT_PIECES = 3;

// three pieces: factors of X C and C^2 in the error of a value, and g' of the exact form
struct split_consts {
    double xc;
    double cc;
    double tiny;  // underflow of the products
    double g_canon;
};

// one piece; FP32 throughout: 1.03 in bf16_split_delta covers the rounding of the bound itself
struct bf16_split_consts {
    float xc;        // factor of X C
    float sum;       // factor of (X + C)^2
    float trunc;     // 2^(IB-23)
    float g_canon;   // g' of the exact-form distance
    int ib;
};

// value error of a row with squared norm at most X2 (Ec = max ||c - bf16(c)||, and ex2 =
// ||x - bf16(x)||^2)
__device__ __forceinline__ float bf16_split_delta(const bf16_split_consts& kc, float X2, float C, float Ec, float ex2) {
    const float X = sqrtf(X2), m = X + C;
    float e = kc.xc * X * C + kc.sum * m * m + 2.4e-7f * (X2 + C * C) + 1e-32f * m + 2e-35f;
    e += 2.0f * (X * Ec + sqrtf(ex2) * C * 1.004f);
    return 1.03f * e;
}

// What the three-piece kernels settle a row by: da the error of its values, and T with every
// centroid that can be the exact-form argmin at or below it (band_threshold, rounded up
// to a float).  in_range: no product or sum of the row passes the float range.
struct split_band {
    double da, T, X2;
    float TF;
    bool in_range;
};
// X = ||x|| and C = max ||c_j||, rounded up
__device__ __forceinline__ split_band make_split_band(const split_consts& kc, double X, double C, float best) {
    split_band b;
    const double m1 = double(best);
    b.X2 = X * X;
    b.da = kc.xc * X * C + kc.cc * C * C + 1e-32 * (X + C) + kc.tiny;
    const double dist_up = fmax(0.0, m1 + b.da + b.X2);
    const double band = (2.0 * b.da + 2.0 * kc.g_canon * dist_up) * (1.0 + 9.5367431640625e-07);
    b.T = m1 + band + (fabs(m1) + b.X2 + C * C) * 4.44e-16;
    b.TF = float(b.T);
    if (double(b.TF) < b.T) b.TF = nextafterf(b.TF, __builtin_inff());
    b.in_range = X < 1e38 && C < 1e38 && 2.0 * X * C + C * C < 1e38 && b.T < 1e38;
    return b;
}
// squared distances: of the centroid with value v at most up, of one with value v or more
// at least lo
__device__ __forceinline__ double split_up(const split_band& b, float v) {
    return double(v) + b.da + b.X2 + (b.X2 + fabs(double(v))) * 1e-15;
}
__device__ __forceinline__ double split_lo(const split_band& b, double v) { return v - b.da + b.X2 * (1.0 - 3e-12); }

// running top-2 of a slot with the first one's index
struct split_slot {
    float m1, m2;
    int id;
    __device__ __forceinline__ void init() {
        m1 = __builtin_inff();
        m2 = __builtin_inff();
        id = 0;
    }
    __device__ __forceinline__ void push(float v, int i) {
        const bool less = v < m1;
        m2 = __builtin_amdgcn_fmed3f(v, m1, m2);
        id = less ? i : id;
        m1 = less ? v : m1;  // not fminf: that takes a second instruction for its operands
    }
};

// bf16 pieces of two floats, packed: first, second and third
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, bf2));
}
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
    p1 = bf16_pair(a, b);
    a -= __uint_as_float(p1 << 16);
    b -= __uint_as_float(p1 & 0xFFFF0000u);
    p2 = bf16_pair(a, b);
    a -= __uint_as_float(p2 << 16);
    b -= __uint_as_float(p2 & 0xFFFF0000u);
    p3 = bf16_pair(a, b);
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

// Blocks of 32 centroids in LDS: a plane of bf16 rows per piece, and 1 KB of norm pieces.
// Three pieces of DP = 128 features are 25 KB a block: three slots, so that two workgroups
// fit a CU; four slots otherwise.
__host__ __device__ constexpr int split_ring(int dp, int pieces) { return dp == 128 && pieces == 3 ? 3 : 4; }
__host__ inline size_t split_lds_bytes(int dp, int pieces) {
    const size_t ring = size_t(split_ring(dp, pieces)) * (size_t(pieces) * 64 * dp + 1024);
    return ring > 16384 ? ring : 16384;  // rows are transposed in it, 4 KB a wave
}

// Workgroup = 4 waves of NB x 32 rows (B operand, every piece in registers for the
// whole pass); blocks of 32 centroids (A operand) stream through the LDS ring by
// direct-to-LDS copies, one barrier per block, as in assign_bf16_kernel.  In a plane,
// 16-byte chunk c of row r sits at chunk c ^ (r % chunks) of its row; at DP = 32, where
// a row is half a 128-byte line, lines of two rows are swizzled by line.  Lane l = 32 h + r
// holds row r's features 32 p + 16 h .. + 15 of every 128-byte piece p of a float row.
// Rows are read as whole 128-byte pieces (eight lanes each, so every load is full
// lines; a lane reading its own row 16 bytes at a time fetched each line from L2 again and
// again: 1.25 ms a launch at n=5e6, d=128, k=512) and pass through the ring's memory to their lanes
// before the ring is filled.  Cs: rows of [c1 DP | c2 DP | c3 DP] bf16 of -2 c_j, and
// cnp: 16 bf16 per row (the norm step's operand), both padded to whole groups of
// four blocks (padding: zero rows with a huge norm).  Slot mb % 4 of a lane takes block
// mb.  Rows without a certain candidate set go to the full list (one piece: to the
// collect rows, for the three-piece kernel).
// The rows' norms are formed here, with three pieces in double: read from a launch of their
// own instead they saved nothing (n=1e7, d=64, k=256: 2.65 and 2.45 ms for all rows, the
// launch 1.2 ms a training).
// Bound: matrix cores (per block and row block 6 DP / 16 + 1 instructions of 32 cycles) and
// about 70 vector instructions of the slots beside them, at two waves a SIMD: n=1e7, d=64,
// k=256 2.5 ms for all rows, the products alone 1.0 ms.  DP = 64 with one row block a wave and
// three waves a SIMD took the same time.  Past a whole group of four blocks, two more are
// enough (k=257: 237 us for n=1e6, d=33, 270 with four).
template <int DP, int NB, int PIECES>
__global__ __launch_bounds__(256, 2) void assign_split_kernel(
    const float* __restrict__ X, int64_t n, int d, const uint16_t* __restrict__ Cs,
    const uint16_t* __restrict__ cnp, int k, const double* __restrict__ cmax_p,
    std::conditional_t<PIECES == 3, split_consts, bf16_split_consts> kc, int32_t* __restrict__ labels, refine_lists L,
    row_select rs) {
    constexpr bool KEYS = PIECES == 1;
    constexpr int HALF = DP / 2;
    constexpr int STEPS = HALF / 8;
    constexpr int LINES = DP / 32;  // 128-byte pieces of a float row
    constexpr int ROWS_PER_WAVE = 32 * NB;
    constexpr int ROWS_PER_WG = 4 * ROWS_PER_WAVE;
    constexpr int CPR = DP / 8;                     // 16-byte chunks of a plane's row
    constexpr int PLANE = 32 * DP * 2;
    constexpr int BLKB = PIECES * PLANE;
    constexpr int NDATA = BLKB / 1024;              // 1 KB copies per block
    constexpr int DPW = (NDATA + 3) / 4;            // of each wave (where they do not divide, some copy the same)
    constexpr int CPW = DPW + 1;                    // + the block's norm pieces
    constexpr int NSL = 4;
    constexpr int RING = split_ring(DP, PIECES);
    constexpr int AHEAD = RING - 1;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int open_cnt[2][4], open_base[2];  // the tile's list entries per wave, and where they go
    unsigned char* ring = smem_raw;                          // [RING][BLKB]
    unsigned char* ring_cn = smem_raw + size_t(RING) * BLKB;  // [RING][1024]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int r32 = lane & 31;
    const int h = lane >> 5;
    // whole groups of four blocks; three pieces: of two
    const int mblocks = KEYS ? bf16_padded_k(k) / 32 : (k + 63) / 64 * 2;
    const int64_t nrows = select_rows(rs, n);
    const int64_t ntiles = (nrows + ROWS_PER_WG - 1) / ROWS_PER_WG;
    // keys
    const float C = float(cmax_p[0]) * (1.0f + 2.4e-7f);
    const float Ec = KEYS ? float(cmax_p[2]) * (1.0f + 2.4e-7f) : 0.f;
    uint32_t kmask = 0, kmv = 0;
    if constexpr (KEYS) {
        kmask = 0x7FFFFFFFu & ~((1u << kc.ib) - 1u);
        asm volatile("v_mov_b32 %0, %1" : "=v"(kmv) : "s"(kmask));
    }

    // this wave's copies of a block (see assign_bf16_kernel): where its 16-byte chunk comes from
    uint32_t voff[DPW], moff[DPW];
#pragma unroll
    for (int c = 0; c < DPW; ++c) {
        const int q = (wave + 4 * c) % NDATA;
        const int p = q * 64 + lane;
        const int plane = p / (PLANE / 16), at = p % (PLANE / 16);
        int row, chunk;
        if constexpr (CPR >= 8) {
            row = at / CPR;
            chunk = (at % CPR) ^ (row & (CPR - 1));
        } else {
            const int line = at >> 3, t = (at & 7) ^ (line & 7);
            row = 2 * line + (t >> 2);
            chunk = t & 3;
        }
        voff[c] = uint32_t(row * (SPLIT_PIECES * DP * 2) + plane * (DP * 2) + chunk * 16);
        moff[c] = lds_addr(ring + q * 1024);
    }
    // byte of chunk c of this lane's row in a plane
    auto chunk_at = [&](int c) {
        if constexpr (CPR >= 8)
            return r32 * (DP * 2) + ((c ^ (r32 & (CPR - 1))) * 16);
        else
            return (r32 >> 1) * 128 + (((((r32 & 1) << 2) | c) ^ ((r32 >> 1) & 7)) * 16);
    };
    const uint32_t voff_cn = uint32_t(lane * 16);
    const uint32_t moff_cn = lds_addr(ring_cn);
    auto issue_block = [&](int mb, int slot) {
        const void* gb = uniform_ptr(reinterpret_cast<const unsigned char*>(Cs) + size_t(mb) * (SPLIT_PIECES * PLANE));
#pragma unroll
        for (int c = 0; c < DPW; ++c) lds_dma16(gb, voff[c], moff[c] + slot * BLKB);
        const void* gc = uniform_ptr(reinterpret_cast<const unsigned char*>(cnp) + size_t(mb) * 1024);
        lds_dma16(gc, voff_cn, moff_cn + slot * 1024);
    };

    // rows of a tile: loaded as floats while the previous tile settles, then split into
    // their pieces, the norm step's operand, and what the settle needs
    uintx4 xp[PIECES][NB][STEPS];
    uintx4 xs_op[NB];
    floatx4 raw[NB][LINES][4];
    int64_t rows[NB];
    double xn[NB];                   // three pieces: ||x|| rounded up
    float x2[NB], xs[NB], da[NB];    // one piece
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
                for (int p = 0; p < LINES; ++p) {
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
            for (int p = 0; p < LINES; ++p) {
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
    // vector q of this lane's row: features 32 (q / 4) + 16 h + 4 (q % 4) ..
    auto features = [&](int nb, int q) {
        floatx4 v = raw[nb][q >> 2][q & 3];
        if (d & 3) {
            const int left = d - 32 * (q >> 2) - 16 * h - 4 * (q & 3);
#pragma unroll
            for (int u = 1; u < 4; ++u) v[u] = u < left ? v[u] : 0.f;
        }
        return v;
    };
    auto split_tile = [&]() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            float sq[4] = {0.f, 0.f, 0.f, 0.f}, se[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 2 * STEPS; ++q) {
                const floatx4 v = features(nb, q);
                if constexpr (KEYS) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) sq[u] = __builtin_fmaf(v[u], v[u], sq[u]);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int s = q >> 1, e = 2 * (q & 1) + u;
                    if constexpr (KEYS) {
                        const uint32_t hi = bf16_pair(v[2 * u], v[2 * u + 1]);
                        xp[0][nb][s][e] = hi;
                        const float e0 = v[2 * u] - __uint_as_float(hi << 16);
                        const float e1 = v[2 * u + 1] - __uint_as_float(hi & 0xFFFF0000u);
                        se[2 * u] = __builtin_fmaf(e0, e0, se[2 * u]);
                        se[2 * u + 1] = __builtin_fmaf(e1, e1, se[2 * u + 1]);
                    } else {
                        uint32_t p1, p2, p3;
                        split_pair(v[2 * u], v[2 * u + 1], p1, p2, p3);
                        xp[0][nb][s][e] = p1;
                        xp[1][nb][s][e] = p2;
                        xp[2][nb][s][e] = p3;
                    }
                }
            }
            // slots: [1 1 1 s_h s_m s_l 0 0] against [c_h c_m c_l 1 1 1 0 0]
            uintx4 op = {0x3F803F80u, 0x00003F80u, 0u, 0u};
            if constexpr (KEYS) {
                // ||x||^2: chains of at most DP / 8 additions, so the relative error is
                // below (DP / 8 + 4) 2^-24
                float t = (sq[0] + sq[1]) + (sq[2] + sq[3]);
                t += __shfl_xor(t, 32);
                x2[nb] = t;
                const float up = t * (1.0f + 2.4e-6f);
                float ex2 = (se[0] + se[1]) + (se[2] + se[3]);
                ex2 = (ex2 + __shfl_xor(ex2, 32)) * (1.0f + 2.4e-6f);
                da[nb] = bf16_split_delta(kc, up, C, Ec, ex2);
                xs[nb] = (up + da[nb]) * (1.0f + 2.4e-7f);
                uint32_t hm, l;
                split3(xs[nb], hm, l);
                op[1] |= hm << 16;
                op[2] = (hm >> 16) | (l << 16);
            } else {
                double t[2] = {0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 2 * STEPS; ++q) {
                    const floatx4 v = features(nb, q);
#pragma unroll
                    for (int u = 0; u < 4; ++u) t[u & 1] = fma(double(v[u]), double(v[u]), t[u & 1]);
                }
                const double sum = t[0] + t[1];
                xn[nb] = sqrt(sum + __shfl_xor(sum, 32)) * (1.0 + 1e-12);
            }
            xs_op[nb] = h == 0 ? op : uintx4{0u, 0u, 0u, 0u};
        }
    };
    load_tile(blockIdx.x);
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        uint32_t m1[NB][NSL], m2[NB][NSL];  // keys
        split_slot st[NB][NSL];             // values
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int q = 0; q < NSL; ++q) {
                m1[nb][q] = 0xFFFFFFFFu;
                m2[nb][q] = 0xFFFFFFFFu;
                st[nb][q].init();
            }
        auto mfma_block = [&](int slot, floatx16(&acc)[NB]) {
            const unsigned char* blk = ring + slot * BLKB;
            auto frag = [&](int piece, int s) {  // step s: features 8 c .. 8 c + 7
                const int c = 4 * (s >> 1) + 2 * h + (s & 1);
                return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uintx4*>(blk + piece * PLANE + chunk_at(c)));
            };
            auto mac = [&](const bf16x8& a, int piece, int s, bool first) {
                const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(bf16x8, xp[piece][nb][s]),
                                                                      first ? zero : acc[nb], 0, 0, 0);
            };
            const bf16x8 an = __builtin_bit_cast(
                bf16x8, *reinterpret_cast<const uintx4*>(ring_cn + slot * 1024 + r32 * 32 + h * 16));
            // the small products first, then x1.c1, then the norms (the error bound
            // counts on this order)
            if constexpr (!KEYS) {
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    const bf16x8 a1 = frag(0, s), a2 = frag(1, s), a3 = frag(2, s);
                    mac(a1, 2, s, s == 0);
                    mac(a3, 0, s, false);
                    mac(a2, 1, s, false);
                    mac(a1, 1, s, false);
                    mac(a2, 0, s, false);
                }
            }
#pragma unroll
            for (int s = 0; s < STEPS; ++s) mac(frag(0, s), 0, s, KEYS && s == 0);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(an, __builtin_bit_cast(bf16x8, xs_op[nb]), acc[nb],
                                                                  0, 0, 0);
        };
        // values of block mb into slot sl (running top-2; keys as in assign_bf16_kernel)
        auto keys_block = [&](const floatx16(&acc)[NB], int mb, int sl) {
            const uint32_t tag = uint32_t(mb) << 4;
            if constexpr (KEYS) {
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
            } else {
                // the register as the index, and the block joined to it once
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const float was = st[nb][sl].m1;
#pragma unroll
                    for (int i = 0; i < 16; ++i) st[nb][sl].push(acc[nb][i], i);
                    st[nb][sl].id = st[nb][sl].m1 < was ? st[nb][sl].id | int(tag) : st[nb][sl].id;
                }
            }
        };
        floatx16 acc0[NB], acc1[NB];
        int slot = 0;  // of block mb
        auto step = [&](int mb, int u, floatx16(&cur)[NB], floatx16(&prev)[NB]) {
            // nothing is scheduled across the wait, the barrier and the copies
            __builtin_amdgcn_sched_barrier(0);
            wait_vm<(AHEAD - 1) * CPW>();
            __syncthreads();
            issue_block(min(mb + AHEAD, mblocks - 1), slot == 0 ? RING - 1 : slot - 1);
            __builtin_amdgcn_sched_barrier(0);
            mfma_block(slot, cur);
            keys_block(prev, mb - 1, (u + 3) & 3);
            slot = slot == RING - 1 ? 0 : slot + 1;
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
        // the first step's "previous block": above every real one
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc1[nb][i] = KEYS ? __uint_as_float(0xFFFFFFFFu) : __builtin_inff();
        int mb = 0;
        for (; mb + 4 <= mblocks; mb += 4) {
            step(mb, 0, acc0, acc1);
            step(mb + 1, 1, acc1, acc0);
            step(mb + 2, 2, acc0, acc1);
            step(mb + 3, 3, acc1, acc0);
        }
        if (!KEYS && mb < mblocks) {
            step(mb, 0, acc0, acc1);
            step(mb + 1, 1, acc1, acc0);
            keys_block(acc1, mblocks - 1, 1);
        } else {
            keys_block(acc1, mblocks - 1, 3);
        }
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
        const int64_t row = nbs ? rows_s[NB - 1] : rows_s[0];
        const bool active = (NB == 2 || h == 0) && row >= 0;
        auto idx_of = [&](uint32_t low, int hh) {
            const int mbk = int(low >> 4), i = int(low & 15u);
            return mbk * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);
        };
        int outcome = 0;  // 1: candidate entry, 2: full entry
        int cnt = 0;
        double other = 0.0;  // bound of the centroids that are not candidates
        int ids[2 * NSL];    // own half's slots, then the partner's: the first's index,
        uint32_t in = 0;     // and which of them are candidates
        if constexpr (KEYS) {
            uint32_t k1[2 * NSL], k2[2 * NSL];
#pragma unroll
            for (int q = 0; q < NSL; ++q) {
                k1[q] = nbs ? m1[NB - 1][q] : m1[0][q];
                k2[q] = nbs ? m2[NB - 1][q] : m2[0][q];
                const uint32_t s1 = (NB == 2 && !h) ? m1[NB - 1][q] : m1[0][q];
                const uint32_t s2 = (NB == 2 && !h) ? m2[NB - 1][q] : m2[0][q];
                k1[NSL + q] = __shfl_xor(s1, 32);
                k2[NSL + q] = __shfl_xor(s2, 32);
            }
            const float X2 = nbs ? x2[NB - 1] : x2[0];
            const float S = nbs ? xs[NB - 1] : xs[0];
            const float dv = nbs ? da[NB - 1] : da[0];
            uint32_t best = 0xFFFFFFFFu;
#pragma unroll
            for (int q = 0; q < 2 * NSL; ++q) {
                best = min(best, k1[q]);
                ids[q] = idx_of(k1[q] & ((1u << kc.ib) - 1u), q < NSL ? h : 1 - h);
            }
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
            int j = 0;
            uint32_t second = 0xFFFFFFFFu;
            bool found = false;
#pragma unroll
            for (int q = 0; q < 2 * NSL; ++q) {
                const bool own = !found && k1[q] == best;
                j = own ? ids[q] : j;
                found = found || own;
                second = min(second, own ? k2[q] : k1[q]);
                cert = cert && k2[q] > TK && (k1[q] > TK || ids[q] < k);
                in |= k1[q] <= TK ? 1u << q : 0u;
            }
            cnt = __popc(in);
            other = double(T) + double(lo_add);
            if (active) {
                if (cert && cnt == 1) {
                    labels[row] = j;
                    if (rs.gap)
                        rs.gap[row] = bound_gap(double(d1), double(__uint_as_float(second & kmask)) + double(lo_add),
                                                rs.gam, rs.base[j]);
                } else {
                    outcome = cert ? 1 : 2;
                }
            }
        } else {
            float v1[2 * NSL], v2[2 * NSL];
#pragma unroll
            for (int q = 0; q < NSL; ++q) {
                const split_slot own = nbs ? st[NB - 1][q] : st[0][q];
                const split_slot to = (NB == 2 && !h) ? st[NB - 1][q] : st[0][q];
                v1[q] = own.m1;
                v2[q] = own.m2;
                ids[q] = idx_of(uint32_t(own.id), h);
                v1[NSL + q] = __shfl_xor(to.m1, 32);
                v2[NSL + q] = __shfl_xor(to.m2, 32);
                ids[NSL + q] = idx_of(uint32_t(__shfl_xor(to.id, 32)), 1 - h);
            }
            float best = v1[0];
#pragma unroll
            for (int q = 1; q < 2 * NSL; ++q) best = v1[q] < best ? v1[q] : best;
            const split_band b = make_split_band(kc, nbs ? xn[NB - 1] : xn[0], cmax_p[0], best);
            bool cert = b.in_range, found = false;
            int j = 0;
            float second = __builtin_inff();
#pragma unroll
            for (int q = 0; q < 2 * NSL; ++q) {
                const bool own = !found && v1[q] == best;
                j = own ? ids[q] : j;
                found = found || own;
                const float v = own ? v2[q] : v1[q];
                second = v < second ? v : second;
                const bool cand = v1[q] <= b.TF;
                cert = cert && v2[q] > b.TF && (!cand || ids[q] < k);
                in |= cand ? 1u << q : 0u;
            }
            cnt = __popc(in);
            other = split_lo(b, b.T);
            if (active) {
                if (cert && cnt == 1) {
                    labels[row] = j;
                    if (rs.gap)
                        rs.gap[row] = bound_gap(split_up(b, best), split_lo(b, double(second)), rs.gam, rs.base[j]);
                } else {
                    outcome = cert && cnt > 0 ? 1 : 2;
                }
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
        if (tid < 2) open_base[tid] = atomicAdd(&L.counters[tid == 0 ? 0 : KEYS ? 2 : 1], tid == 0 ? tc : tl);
        __syncthreads();
        int e0 = open_base[0], f0 = open_base[1];
        for (int w = 0; w < wave; ++w) {
            e0 += open_cnt[0][w];
            f0 += open_cnt[1][w];
        }
        if (outcome == 1) {
            const int e = e0 + lanes_below(mc);
            L.cand_rows[e] = int32_t(row);
            L.cand_count[e] = cnt;
            if (rs.gap) L.cand_lo[e] = float_below(other);
            int c = 0;
#pragma unroll
            for (int q = 0; q < 2 * NSL; ++q)
                if ((in >> q) & 1u) L.cand_ids[int64_t(e) * MAXC + c++] = ids[q];
        }
        if (outcome == 2) (KEYS ? L.coll_rows : L.full_rows)[f0 + lanes_below(ml)] = int32_t(row);
    }
}

}  // namespace km
