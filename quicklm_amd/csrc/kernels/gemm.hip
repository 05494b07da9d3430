// int8 weight-only matmul for M > 1 on the gfx950 matrix cores:
//   y[m, n] = sum_k x[m, k] * q[n, k] * s[n, k / G]
// Replaces math::matmul's int8 branch with M > 1 (reference
// math_ops.cpp:845-871: batched decode M = B, prefill M = T - 1).
//
// Arithmetic. The int8 weights are exact in bf16 (|q| <= 127 fits the 8-bit
// significand). Each activation is split into bf16 hi + lo (hi = RNE(x),
// lo = RNE(x - hi)), so hi + lo carries 16 significant bits and the only
// rounding left is |x - hi - lo| <= 2^-17 |x|; the products and sums run in
// fp32 inside the bf16 MFMAs. The MFMAs of a 32-column group (hi and lo) start
// from zero and the result tile is scaled by s[n, group] in fp32 and
// accumulated, so the weights are never rounded. Per-row scales (G = K) chain
// the MFMAs and scale once at the end. Normwise error vs the fp32 reference
// is ~1e-6.
//
// M <= 64 (batched decode): k_mm_i8_sk, weight streaming with K split across
// workgroups. More rows (prefill), and bf16 weight rows from 17: k_mm_pf over
// an activation split once per call. Epilogues: store, residual add, SwiGLU
// (weights [2F, K]: silu(gate) * up formed in registers).

#include <algorithm>

#include "common.hpp"
#include "mm_reduce.hpp"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
enum { EPI_STORE = 0, EPI_RESID = 1, EPI_SWIGLU = 2 };

__device__ __forceinline__ unsigned bf16_rne_bits(float x) {
    unsigned u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}

// hi/lo bf16 pair of x packed as (hi, lo) 16-bit halves
__device__ __forceinline__ void split_bf16(float x, unsigned short& hi, unsigned short& lo) {
    const unsigned h = bf16_rne_bits(x);
    hi = (unsigned short)h;
    lo = (unsigned short)bf16_rne_bits(x - __uint_as_float(h << 16));
}

// int8 -> bf16 bits (exact): the float's upper half
__device__ __forceinline__ unsigned short i8_bf16(int v) {
    return (unsigned short)(__float_as_uint((float)v) >> 16);
}

__device__ __forceinline__ unsigned i8_bf16x2(int lo, int hi) {
    // the upper halves of the two floats, in one byte permute
    return __builtin_amdgcn_perm(__float_as_uint((float)hi), __float_as_uint((float)lo),
                                 0x07060302u);
}

// RMSNorm of a staged activation: (x * s) * (1 + w), the reference's order
// (math_ops.cpp:1021-1031), s = 1/sqrt(mean(x^2) + eps) of the row.
__device__ __forceinline__ float4 norm4(float4 v, float s, float4 w) {
    v.x = (v.x * s) * (1.0f + w.x);
    v.y = (v.y * s) * (1.0f + w.y);
    v.z = (v.z * s) * (1.0f + w.z);
    v.w = (v.w * s) * (1.0f + w.w);
    return v;
}

__device__ __forceinline__ void store_hilo(unsigned short* hi, unsigned short* lo, float4 v) {
    unsigned short h[4], l[4];
    split_bf16(v.x, h[0], l[0]);
    split_bf16(v.y, h[1], l[1]);
    split_bf16(v.z, h[2], l[2]);
    split_bf16(v.w, h[3], l[3]);
    *reinterpret_cast<uint2*>(hi) = make_uint2((unsigned)h[0] | ((unsigned)h[1] << 16),
                                               (unsigned)h[2] | ((unsigned)h[3] << 16));
    *reinterpret_cast<uint2*>(lo) = make_uint2((unsigned)l[0] | ((unsigned)l[1] << 16),
                                               (unsigned)l[2] | ((unsigned)l[3] << 16));
}

// 16 int8 -> 16 bf16 (exact), as two 16-byte LDS stores
__device__ __forceinline__ void store_w16(unsigned short* dst, int4 w) {
    const int wv[4] = {w.x, w.y, w.z, w.w};
    uint4 o[2];
    unsigned* ow = reinterpret_cast<unsigned*>(o);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const unsigned v = (unsigned)wv[j];
        const int b0 = (int8_t)(v & 0xffu), b1 = (int8_t)((v >> 8) & 0xffu);
        const int b2 = (int8_t)((v >> 16) & 0xffu), b3 = (int8_t)(v >> 24);
        ow[2 * j] = (unsigned)i8_bf16(b0) | ((unsigned)i8_bf16(b1) << 16);
        ow[2 * j + 1] = (unsigned)i8_bf16(b2) | ((unsigned)i8_bf16(b3) << 16);
    }
    reinterpret_cast<uint4*>(dst)[0] = o[0];
    reinterpret_cast<uint4*>(dst)[1] = o[1];
}

// Tile-major weights (qlm_mx_swizzle: 16-row x 64-column fragments of 1 KB
// in lane order, each half of a [gate; up] matrix tiled on its own; group-32
// scales as [fragment][h][n]). Row r of the stacked matrix is row r - half F
// of half `half`; its 16 columns k .. k + 15 (k a multiple of 16) are one
// lane's 16 bytes of fragment (tile, k / 64). Per-row scales keep their
// [rows] layout.
struct TileMap {
    int F;           // rows per half (all rows when the matrix has one half)
    int tiles_half;  // 16-row tiles per half
    int nblk64;      // 64-column blocks per row
};
__device__ __forceinline__ int tm_frag(const TileMap& t, int r, int k, int& n) {
    const int half = r >= t.F ? 1 : 0;
    const int rh = r - half * t.F;
    n = rh & 15;
    return (half * t.tiles_half + (rh >> 4)) * t.nblk64 + (k >> 6);
}
// byte offset of row r's 16 columns k .. k + 15
__device__ __forceinline__ size_t tm_off(const TileMap& t, int r, int k) {
    int n;
    const int fb = tm_frag(t, r, k, n);
    return ((size_t)fb * 64 + ((k >> 4) & 3) * 16 + n) * 16;
}
// index of row r's scale for the 32-column group g
__device__ __forceinline__ size_t tm_scale(const TileMap& t, int r, int g) {
    int n;
    const int fb = tm_frag(t, r, g * 32, n);
    return (size_t)fb * 32 + (g & 1) * 16 + n;
}

// bf16 weight rows with a workspace too small for the split activation: each
// workgroup of 4 waves (2 x 2, 64 rows x 64 weight rows each) converts the
// activation chunks it stages itself, and applies the RMSNorm there (NORM).
// KG: 32-column groups per staged chunk.
template <int EPI, bool NORM, int KG>
__global__ __launch_bounds__(kThreads) void k_mm_bf16(const float* __restrict__ x, int ldx,
                                                      const float* __restrict__ rs,
                                                      const float* __restrict__ nw,
                                                      const uint16_t* __restrict__ w,
                                                      float* __restrict__ y, int ldy, int M,
                                                      int N, int K) {
    constexpr int TM = 4, TN = 4, BM = 128, BN = 128;
    constexpr int KC = 32 * KG;
    constexpr int XP = KC + 8;        // padded LDS rows (bf16 elements)
    constexpr int XPT = BM * KC / 4 / kThreads;   // float4 per thread and x chunk
    constexpr int WPT = BN * KC / 16 / kThreads;  // 32 bytes per thread and weight chunk
    constexpr int OUT_TN = EPI == EPI_SWIGLU ? TN / 2 : TN;  // output tiles per wave
    constexpr int BN_OUT = 2 * OUT_TN * 16;                   // output columns per workgroup
    __shared__ __attribute__((aligned(16))) unsigned short xs_hi[BM * XP], xs_lo[BM * XP],
        ws[BN * XP];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wn = wave & 1, wm = wave >> 1;
    const int m0 = blockIdx.y * BM;
    const int nout0 = blockIdx.x * BN_OUT;  // first output column of the workgroup

    // staged weight row r -> global weight row (clamped into the matrix)
    auto w_row = [&](int r) -> int {
        if constexpr (EPI == EPI_SWIGLU) {
            const int half = BN / 2;
            return r < half ? min(nout0 + r, N - 1) : N + min(nout0 + (r - half), N - 1);
        } else {
            return min(nout0 + r, N - 1);
        }
    };
    // a wave's tile tn -> first staged row of that tile
    auto tile_row = [&](int tn) -> int {
        if constexpr (EPI == EPI_SWIGLU)
            return tn < TN / 2 ? (wn * (TN / 2) + tn) * 16
                               : BN / 2 + (wn * (TN / 2) + tn - TN / 2) * 16;
        else
            return (wn * TN + tn) * 16;
    };

    float4 xr[XPT];
    float4 gr[NORM ? XPT : 1];  // RMSNorm gain of the same columns
    float rr[NORM ? XPT : 1];   // RMSNorm row scale
    int4 wr[WPT][2];
    auto load_chunk = [&](int c) {
        const int k0 = c * KC;
#pragma unroll
        for (int u = 0; u < XPT; ++u) {
            const int i = tid + u * kThreads;
            const int r = i / (KC / 4), c4 = i % (KC / 4);
            const int m = min(m0 + r, M - 1);
            xr[u] = *reinterpret_cast<const float4*>(x + (size_t)m * ldx + k0 + c4 * 4);
            if constexpr (NORM) {
                gr[u] = *reinterpret_cast<const float4*>(nw + k0 + c4 * 4);
                rr[u] = rs[m];
            }
        }
#pragma unroll
        for (int u = 0; u < WPT; ++u) {
            const int i = tid + u * kThreads;
            const int r = i / (KC / 16), c16 = i % (KC / 16);
            const int4* p =
                reinterpret_cast<const int4*>(w + (size_t)w_row(r) * K + k0 + c16 * 16);
            wr[u][0] = p[0];
            wr[u][1] = p[1];
        }
    };
    auto store_chunk = [&]() {
#pragma unroll
        for (int u = 0; u < XPT; ++u) {
            const int i = tid + u * kThreads;
            const int r = i / (KC / 4), c4 = i % (KC / 4);
            float4 v = xr[u];
            if constexpr (NORM) v = norm4(v, rr[u], gr[u]);
            store_hilo(&xs_hi[r * XP + c4 * 4], &xs_lo[r * XP + c4 * 4], v);
        }
#pragma unroll
        for (int u = 0; u < WPT; ++u) {
            const int i = tid + u * kThreads;
            const int r = i / (KC / 16), c16 = i % (KC / 16);
            int4* dst = reinterpret_cast<int4*>(&ws[r * XP + c16 * 16]);
            dst[0] = wr[u][0];
            dst[1] = wr[u][1];
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int nch = K / KC;
    load_chunk(0);
    for (int c = 0; c < nch; ++c) {
        __syncthreads();  // the previous chunk's LDS reads are done
        store_chunk();
        __syncthreads();
        if (c + 1 < nch) load_chunk(c + 1);
#pragma unroll
        for (int gg = 0; gg < KG; ++gg) {
            const int kofs = gg * 32 + (lane >> 4) * 8;
            bf16x8 ah[TM], al[TM], bw[TN];
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) {
                const int r = (wm * TM + tm) * 16 + (lane & 15);
                ah[tm] = *reinterpret_cast<const bf16x8*>(&xs_hi[r * XP + kofs]);
                al[tm] = *reinterpret_cast<const bf16x8*>(&xs_lo[r * XP + kofs]);
            }
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
                bw[tn] = *reinterpret_cast<const bf16x8*>(
                    &ws[(tile_row(tn) + (lane & 15)) * XP + kofs]);
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) {
                    acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[tm], bw[tn],
                                                                         acc[tm][tn], 0, 0, 0);
                    acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[tm], bw[tn],
                                                                         acc[tm][tn], 0, 0, 0);
                }
        }
    }

    // ---- epilogue: lane holds rows (lane/16)*4 + i, column lane%16 of each tile ----
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < OUT_TN; ++tn) {
            const int n = nout0 + (wn * OUT_TN + tn) * 16 + (lane & 15);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + (wm * TM + tm) * 16 + (lane >> 4) * 4 + i;
                if (m < M && n < N) {
                    float* dst = y + (size_t)m * ldy + n;
                    if constexpr (EPI == EPI_SWIGLU)
                        *dst = silu_f(acc[tm][tn][i]) * acc[tm][tn + TN / 2][i];
                    else if constexpr (EPI == EPI_RESID)
                        *dst += acc[tm][tn][i];
                    else
                        *dst = acc[tm][tn][i];
                }
            }
        }
}

// ---------------------------------------------------------------------------
// Many rows (prefill): weights of any stored form (WK) against the pre-split
// activation (k_split_op): 128 activation rows x 256 staged weight rows a
// workgroup (SwiGLU: 128 gate and the matching 128 up rows), four waves of
// 64 x 128 each, two workgroups a CU.
//   - Operands sit in LDS as 32 x 16 MFMA operands of 1 KB in lane order (lane
//     l's 16 bytes at 16 l: row l & 31, columns 8 (l >> 5) .. + 7), so every
//     ds_read_b128 is lane-contiguous; the activation comes from global memory
//     in that order already. A 64 x 128 wave tile reads 16 KB of them a
//     32-column group for 32 MFMAs of 32 cycles; the 64 x 64 tile before it
//     read 12 KB for half as many, and LDS bound it.
//   - Two stages, one barrier per 32-column group: group g + 1 is converted and
//     stored while group g is multiplied, and group g + 2 requested. Buffer
//     loads (uniform base, scalar group offset, 32-bit lane offset) leave no
//     address arithmetic in the loop; group scales go through LDS.
//   - Every load is unconditional (clamped rows, tiles and groups).
// Group-32 scales: a group's four MFMAs (two k-steps, hi and lo) start from
// zero and the 32 x 32 result is scaled into the sum in fp32, so the weights
// are never rounded; one scale a row, or bf16 weights: the MFMAs chain over K.
// PART: the sums of one K slice go to part[slice][m][NR] (k_mm_reduce adds
// them in slice order and applies the epilogue).
// Bound by the matrix cores and the vector work beside them: 2048 rows, 4B
// gate/up (2 x 9728 x 2560) 493 -> 388 us with int8 groups (1050 TFLOP/s with
// hi and lo counted; a large bf16 library product reaches 1384 on the same
// card), 390 -> 336 us with row scales, 437 -> 339 us with bf16 rows. Measured
// and not kept: all scale FMAs of a tile right after its products (414 us),
// 64-bit lane addresses (spills, 605 us), activation registers reloaded half
// a group ahead for bf16 rows too (413 us).
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
enum { W_TILES = 0, W_ROWS = 1, W_BF16 = 2 };
constexpr int kPfM = 128, kPfN = 256;  // staged rows of a workgroup
constexpr int kPfBlocks = 512;         // most workgroups of a sliced launch

// Buffer descriptor of a uniform base: a load then takes a lane's 32-bit
// offset and a scalar one, no vector arithmetic on addresses.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0, -1, 0x00027000);
}

struct PfArgs {
    const uint16_t* xs;  // split activation: hi plane, lo plane M * K further
    const void* q;
    const float* sc;
    float* y;  // output, or the slices' partial sums
    int ldy, M, N, K;
    int gx, gy, blocks;  // column blocks, row blocks, blocks in all (slices included)
    int gslice;          // 32-column groups a slice
};

template <int WK, bool RS, int EPI, bool PART>
__global__ __launch_bounds__(256, 2) void k_mm_pf(const PfArgs a) {
    constexpr bool SWIGLU = EPI == EPI_SWIGLU;
    constexpr bool I8 = WK != W_BF16;
    constexpr bool GS = I8 && !RS;
    constexpr int BN_OUT = SWIGLU ? kPfN / 2 : kPfN;
    constexpr int BS = I8 ? 2 : 4;  // 16-byte weight loads a thread and group
    constexpr int A_LO = 8192, B_OFS = 16384, S_OFS = 32768, STAGE = 32768 + (GS ? 1024 : 0);
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // Workgroups go to the 8 XCDs in turn: XCD i takes the i-th eighth of the
    // blocks, in bands of 8 row blocks (column by column inside a band), so
    // the 64 workgroups an XCD holds read about 8 row blocks x 8 column
    // blocks of operands through its L2.
    const int per = (a.blocks + 7) >> 3;
    int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (t >= a.blocks) return;
    const int area = a.gx * a.gy;
    const int slice = t / area;
    t -= slice * area;
    const int band = t / (8 * a.gx);
    const int bh = min(8, a.gy - 8 * band);
    t -= band * 8 * a.gx;
    const int m0 = (8 * band + t % bh) * kPfM;
    const int nout0 = (t / bh) * BN_OUT;
    const int M = a.M, N = a.N, K = a.K;
    const int ngrp = K >> 5;
    const int g0 = slice * a.gslice, g1 = min(ngrp, g0 + a.gslice);

    // staged 16-row weight tile t16 (0..15) -> first matrix row / tile-major tile
    const int tiles_half = (N + 15) >> 4;
    auto tile_of = [&](int t16, int& half) -> int {
        half = SWIGLU ? t16 >> 3 : 0;
        return min((nout0 >> 4) + (SWIGLU ? t16 & 7 : t16), tiles_half - 1);
    };
    // matrix row of staged row n of tile t16 (clamped)
    auto row_of = [&](int t16, int n) -> int {
        int half;
        const int tl = tile_of(t16, half);
        return half * N + min(tl * 16 + n, N - 1);
    };
    // a wave's 32-row tile tn -> staged 32-row tile
    auto t32_of = [&](int tn) -> int {
        return SWIGLU ? (tn >> 1) * 4 + wn * 2 + (tn & 1) : wn * 4 + tn;
    };

    // Uniform bases advance by constants a group; a lane adds its 32-bit offset.
    // Activation: slot tid + 256 u of 4 tiles x 4 octets x 32 rows, as in LDS.
    // In a plane tile T's rows are stored [octet][row][8], R = min(32, M - 32 T)
    // rows a tile.
    const int mt_last = (M - 1) >> 5;
    const char* ab[2];
    int astep[2];
    unsigned ao[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int T = min((m0 >> 5) + 2 * u + (wave >> 1), mt_last);
        const int R = min(32, M - 32 * T);
        astep[u] = 64 * R;
        ab[u] = reinterpret_cast<const char*>(a.xs) + (size_t)T * 64 * K + (size_t)g0 * astep[u];
        ao[u] = (unsigned)((((tid >> 5) & 3) * R + min(tid & 31, R - 1)) * 16);
    }
    const size_t plane = (size_t)M * K * 2;
    // Weights. int8: slot tid + 256 u of 16 tiles x 2 k-steps x 16 rows, 16
    // columns each; bf16: slot tid + 256 u of 256 rows x 4 octets. Load u
    // stays inside one half of a [gate; up] matrix.
    constexpr int TU = 16 / BS;  // 16-row tiles a load
    const char* bb[BS];
    unsigned bo[BS];
#pragma unroll
    for (int u = 0; u < BS; ++u) {
        int half, h2;
        const int tl0 = tile_of(TU * u, half);
        if constexpr (WK == W_TILES) {
            bb[u] = static_cast<const char*>(a.q) +
                    (size_t)(half * tiles_half + tl0) * (K >> 6) * 1024 + (size_t)512 * g0;
            bo[u] = (unsigned)(tile_of(TU * u + (tid >> 5), h2) - tl0) * (unsigned)((K >> 6) * 1024) +
                    (tid & 31) * 16;
        } else if constexpr (WK == W_ROWS) {
            const int r0 = row_of(TU * u, 0);
            bb[u] = static_cast<const char*>(a.q) + (size_t)r0 * K + (size_t)32 * g0;
            bo[u] = (unsigned)(row_of(TU * u + (tid >> 5), tid & 15) - r0) * (unsigned)K +
                    ((tid >> 4) & 1) * 16;
        } else {
            const int r0 = row_of(TU * u, 0);
            bb[u] = static_cast<const char*>(a.q) + ((size_t)r0 * K + (size_t)32 * g0) * 2;
            bo[u] = ((unsigned)(row_of(TU * u + (tid >> 6), (tid >> 2) & 15) - r0) * (unsigned)K +
                     (tid & 3) * 8) * 2;
        }
    }
    constexpr int BSTEP = WK == W_TILES ? 512 : WK == W_ROWS ? 32 : 64;
    // group scales: thread tid takes staged row tid's
    const char* sb = nullptr;
    unsigned so = 0;
    if constexpr (GS) {
        // the first lane's tile is the base (a wave's rows lie in one half)
        int half, h2;
        const int tl0 = tile_of(4 * wave, half);
        if constexpr (WK == W_TILES) {
            sb = reinterpret_cast<const char*>(
                a.sc + (size_t)(half * tiles_half + tl0) * (K >> 6) * 32 + (size_t)16 * g0);
            so = ((unsigned)(tile_of(tid >> 4, h2) - tl0) * (unsigned)((K >> 6) * 32) +
                  (tid & 15)) * 4;
        } else {
            const int r0 = row_of(4 * wave, 0);
            sb = reinterpret_cast<const char*>(a.sc + (size_t)r0 * ngrp + g0);
            so = (unsigned)(row_of(tid >> 4, tid & 15) - r0) * (unsigned)ngrp * 4;
        }
    }
    constexpr int SSTEP = WK == W_TILES ? 64 : 4;

    constexpr int XR = GS ? 1 : 2;  // sets of activation staging registers
    u32x4 xh[XR], xl[XR], wb[BS];
    float sl = 0.0f;
    // i: group - g0
    __amdgpu_buffer_rsrc_t bd[BS], xhd[2], xld[2];
    const __amdgpu_buffer_rsrc_t sd = make_rsrc(sb);
#pragma unroll
    for (int u = 0; u < BS; ++u) bd[u] = make_rsrc(bb[u]);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        xhd[u] = make_rsrc(ab[u]);
        xld[u] = make_rsrc(ab[u] + plane);
    }
    auto load_w = [&](int i, int u) {
        wb[u] = __builtin_amdgcn_raw_buffer_load_b128(bd[u], bo[u], BSTEP * i, 0);
    };
    auto load_s = [&](int i) {
        if constexpr (GS)
            sl = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(sd, so, SSTEP * i, 0));
    };
    auto load_x = [&](int i, int u) {
        xh[u % XR] = __builtin_amdgcn_raw_buffer_load_b128(xhd[u], ao[u], i * astep[u], 0);
        xl[u % XR] = __builtin_amdgcn_raw_buffer_load_b128(xld[u], ao[u], i * astep[u], 0);
    };
    // int8 slot u: 16 int8 -> 16 bf16 (exact), two words of four a call;
    // columns 0-7 of a k-step (words 0, 1), then 8-15. bf16: row r, octet o at
    // slot r ^ 4 o of its octet, so that a wave's 16 rows x 4 octets meet no
    // bank twice in a phase
    unsigned ow[4];
    auto convert = [&](int u, int word) {
        const unsigned v = wb[u][word];
        ow[2 * (word & 1)] = i8_bf16x2((int8_t)(v & 0xffu), (int8_t)((v >> 8) & 0xffu));
        ow[2 * (word & 1) + 1] = i8_bf16x2((int8_t)((v >> 16) & 0xffu), (int8_t)(v >> 24));
    };
    auto store_w = [&](unsigned char* st, int u, int oct) {
        const int s = tid + 256 * u;
        if constexpr (I8) {
            *reinterpret_cast<u32x4*>(st + B_OFS + (s >> 6) * 2048 + ((s >> 4) & 1) * 1024 +
                                      (((s >> 5) & 1) * 16 + (s & 15)) * 16 + oct * 512) =
                u32x4{ow[0], ow[1], ow[2], ow[3]};
        } else {
            const int o = s & 3, r = (s >> 2) & 31;
            *reinterpret_cast<u32x4*>(st + B_OFS + (s >> 7) * 2048 + o * 512 + (r ^ (4 * o)) * 16) =
                wb[u];
        }
    };
    auto store_x = [&](unsigned char* st, int u) {
        *reinterpret_cast<u32x4*>(st + (tid + 256 * u) * 16) = xh[u % XR];
        *reinterpret_cast<u32x4*>(st + A_LO + (tid + 256 * u) * 16) = xl[u % XR];
    };
    auto store_s = [&](unsigned char* st) {
        if constexpr (GS) *reinterpret_cast<float*>(st + S_OFS + tid * 4) = sl;
    };

    f32x16 acc[2][4];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int tn = 0; tn < 4; ++tn)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[tm][tn][i] = 0.0f;

    const int ng = g1 - g0;
    for (int u = 0; u < BS; ++u) load_w(0, u);
    load_s(0);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        load_x(0, u);
        store_x(smem, u);
    }
#pragma unroll
    for (int u = 0; u < BS; ++u) {
        if constexpr (I8) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                convert(u, 2 * h);
                convert(u, 2 * h + 1);
                store_w(smem, u, h);
            }
        } else {
            store_w(smem, u, 0);
        }
    }
    store_s(smem);
    const int i1 = min(1, ng - 1);
    for (int u = 0; u < BS; ++u) load_w(i1, u);
    load_s(i1);
    if constexpr (XR == 2) {
        load_x(i1, 0);
        load_x(i1, 1);
    }
    __syncthreads();

    // The scale FMAs of tile j run under the matrix instructions of tile j + 1
    // (tile 7's under the next group's first), the conversions under the rest:
    // the order is fixed by scheduling fences, which the compiler's own order
    // (all FMAs of a tile after its products) would serialise.
    f32x16 d[2];
    float s_cur[4], s_prev = 0.0f;
    if constexpr (GS) {
#pragma unroll
        for (int e = 0; e < 16; ++e) d[1][e] = 0.0f;
    }
#pragma unroll 1
    for (int i = 0; i < ng; ++i) {
        const unsigned char* st = smem + (i & 1) * STAGE;
        // group i + 1 goes into the other stage (its last reads ended at the
        // previous barrier); past the end a copy of the last group nobody reads
        unsigned char* nx = smem + ((i + 1) & 1) * STAGE;
        const int ix = min(i + 1, ng - 1), i2 = min(i + 2, ng - 1);
        bf16x8 ah[2][2], al[2][2], bw[2];  // [tile][k-step]
        auto read_b = [&](int tn, int k) {
            const unsigned char* p = st + B_OFS + t32_of(tn) * 2048;
            if constexpr (I8) {
                p += k * 1024 + lane * 16;
            } else {
                const int o = 2 * k + (lane >> 5);
                p += o * 512 + ((lane & 31) ^ (4 * o)) * 16;
            }
            bw[k] = *reinterpret_cast<const bf16x8*>(p);
        };
        auto read_s = [&](int tn) {
            if constexpr (GS)
                s_cur[tn] = *reinterpret_cast<const float*>(st + S_OFS +
                                                            (t32_of(tn) * 32 + (lane & 31)) * 4);
        };
        auto read_a = [&](int tm, int k) {
            const unsigned char* p = st + (wm * 2 + tm) * 2048 + k * 1024 + lane * 16;
            ah[tm][k] = *reinterpret_cast<const bf16x8*>(p);
            al[tm][k] = *reinterpret_cast<const bf16x8*>(p + A_LO);
        };
        read_b(0, 0);
        read_a(0, 0);
        read_b(0, 1);
        read_a(0, 1);
        read_a(1, 0);
        read_a(1, 1);
        read_s(0);
        if constexpr (XR == 1) load_x(ix, 0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int tn = j >> 1, tm = j & 1;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int k = kk >> 1;
                const bf16x8 av = kk & 1 ? al[tm][k] : ah[tm][k];
                if constexpr (GS) {
                    if (kk == 0) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) d[j & 1][e] = 0.0f;
                    }
                    d[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bw[k], d[j & 1],
                                                                      0, 0, 0);
                } else {
                    acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bw[k],
                                                                         acc[tm][tn], 0, 0, 0);
                }
                // the next column tile's weights
                if (tn < 3 && tm == 1 && (kk & 1)) read_b(tn + 1, k);
                if (tn < 3 && tm == 1 && kk == 2) read_s(tn + 1);
                if (GS && kk > 0) {
                    const int p = (j + 7) & 7, pn = p >> 1, pm = p & 1;
                    const float sv = j == 0 ? s_prev : s_cur[pn];
#pragma unroll
                    for (int e = kk == 1 ? 0 : kk == 2 ? 5 : 10; e < (kk == 1 ? 5 : kk == 2 ? 10 : 16);
                         ++e)
                        acc[pm][pn][e] = fmaf(d[p & 1][e], sv, acc[pm][pn][e]);
                }
                // staging: weights word by word from tile 2 on, each register
                // reloaded as soon as it is stored, so that a load has about
                // three quarters of a group to return
                if constexpr (I8) {
                    const int step = (j - 2) * 2 + (kk >> 1);  // 0..11 over tiles 2..7
                    if (j >= 2 && (kk == 0 || kk == 2) && step % 3 != 2) {
                        const int w = step / 3 * 2 + step % 3;  // 0..7
                        convert(w >> 2, w & 3);
                        if (w & 1) store_w(nx, w >> 2, (w >> 1) & 1);
                        if ((w & 3) == 3) load_w(i2, w >> 2);
                    }
                    if (j == 2 && kk == 1) {
                        store_s(nx);
                        load_s(i2);
                    }
                } else if (kk == 1 && j >= 2 && j < 2 + BS) {
                    store_w(nx, j - 2, 0);
                    load_w(i2, j - 2);
                }
                if constexpr (XR == 1) {
                    if (j == 4 && kk == 0) {
                        store_x(nx, 0);
                        load_x(ix, 1);
                    }
                    if (j == 7 && kk == 3) store_x(nx, 1);
                } else if (kk == 3 && (j == 3 || j == 6)) {
                    store_x(nx, j == 6);
                    load_x(i2, j == 6);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (GS) s_prev = s_cur[3];
        __syncthreads();
    }
    if constexpr (GS) {
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[1][3][e] = fmaf(d[1][e], s_prev, acc[1][3][e]);
    }
    // a wave whose rows or columns all lie outside the matrix only staged
    const bool busy = m0 + wm * 64 < M && nout0 + wn * (BN_OUT / 2) < N;
    if (!busy) return;

    // lane l of a 32 x 32 tile: column l & 31, rows 8 (e >> 2) + 4 (l >> 5) + (e & 3)
    if constexpr (I8 && RS) {
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) {
            const float s = a.sc[row_of(2 * t32_of(tn) + ((lane >> 4) & 1), lane & 15)];
#pragma unroll
            for (int tm = 0; tm < 2; ++tm)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[tm][tn][e] *= s;
        }
    }
    constexpr int OUT_TN = SWIGLU && !PART ? 2 : 4;
    const int NR = SWIGLU ? 2 * N : N;
    const int mw = m0 + wm * 64 + 4 * (lane >> 5);
#pragma unroll
    for (int tn = 0; tn < OUT_TN; ++tn) {
        const int half = SWIGLU ? tn >> 1 : 0;
        const int n = nout0 + (SWIGLU ? (wn * 2 + (tn & 1)) * 32 : t32_of(tn) * 32) + (lane & 31);
        if (n >= N) continue;
        // the residuals of a column tile are requested together: one load
        // before each store would be a round trip to memory an element
        // (out-projection, 2048 rows and columns: 108 against 78 us)
        float rv[2][16];
        if constexpr (EPI == EPI_RESID && !PART) {
#pragma unroll
            for (int tm = 0; tm < 2; ++tm)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    rv[tm][e] = a.y[(size_t)min(mw + tm * 32 + 8 * (e >> 2) + (e & 3), M - 1) *
                                        a.ldy + n];
        }
#pragma unroll
        for (int tm = 0; tm < 2; ++tm)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = mw + tm * 32 + 8 * (e >> 2) + (e & 3);
                if (m >= M) continue;
                const float v = acc[tm][tn][e];
                if constexpr (PART)
                    a.y[((size_t)slice * M + m) * NR + half * N + n] = v;
                else if constexpr (SWIGLU)
                    a.y[(size_t)m * a.ldy + n] = silu_f(v) * acc[tm][tn + 2][e];
                else if constexpr (EPI == EPI_RESID)
                    a.y[(size_t)m * a.ldy + n] = rv[tm][e] + v;
                else
                    a.y[(size_t)m * a.ldy + n] = v;
            }
    }
}

// ---------------------------------------------------------------------------
// M <= 64 (batched decode): weight streaming with K split across workgroups.
//
// A workgroup owns 64 weight rows (wave w: rows 16w..16w+15 as one MFMA
// n-tile) and 16*TM activation rows, over a K slice of kper columns; per
// 128-column chunk (4 groups) x [BM, 128] is staged as bf16 hi/lo (with the
// RMSNorm applied when NORM) and the weights [64, 128] as bf16, the next
// chunk being loaded into registers meanwhile. Each slice writes its fp32
// partial tile to part[ks, m, n]; k_mm_reduce sums the slices in order and
// applies the epilogue. With a single slice and a plain store the partial
// is the output itself.
constexpr int kSkRows = 64;
constexpr int kSkKc = 128;
// chunks in flight per workgroup (register ring), by activation tiles
constexpr int sk_ring(int tm) { return tm <= 2 ? 2 : 1; }

// DEFER (with NORM): the activation is staged as x * (1 + w) and the row's
// 1/rms multiplies the reduced sums instead (k_mm_reduce<..., true>), so no
// separate row-scale launch precedes the matmul.
// TL: q and sc are tile-major (TileMap tmap); otherwise row-major.
template <int TM, bool ROWSCALE, bool NORM, bool DEFER, bool TL = false>
__global__ __launch_bounds__(kThreads) void k_mm_i8_sk(
    const float* __restrict__ x, int ldx, const float* __restrict__ rs,
    const float* __restrict__ nw, const int8_t* __restrict__ q, const float* __restrict__ sc,
    float* __restrict__ part, int ldp, int M, int NR, int K, int kper, TileMap tmap) {
    constexpr int BM = 16 * TM;
    constexpr int KC = kSkKc;
    constexpr int XP = KC + 8, WP = KC + 8;
    constexpr int XV = BM * KC / 4, WV = kSkRows * KC / 16;
    constexpr int XPT = (XV + kThreads - 1) / kThreads;
    constexpr int WPT = (WV + kThreads - 1) / kThreads;
    constexpr int CPF = sk_ring(TM);
    __shared__ __attribute__((aligned(16))) unsigned short xs_hi[BM * XP];
    __shared__ __attribute__((aligned(16))) unsigned short xs_lo[BM * XP];
    __shared__ __attribute__((aligned(16))) unsigned short ws[kSkRows * WP];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = blockIdx.x * kSkRows;
    const int ks = blockIdx.y;
    const int m0 = blockIdx.z * BM;
    const int kb = ks * kper;
    const int nblk = K >> 5;
    const int ncol = n0 + wave * 16 + (lane & 15);      // this lane's weight row (output column)
    const int nrow = ncol < NR ? ncol : NR - 1;

    // a ring of CPF chunk buffers in registers: a chunk's registers are
    // refilled with chunk c + CPF as soon as chunk c is staged to LDS, so a
    // workgroup's whole K slice (<= CPF chunks) is requested at once
    float4 xr[CPF][XPT];
    float4 gr[CPF][NORM ? XPT : 1];
    float rr[CPF][NORM ? XPT : 1];
    int4 wr[CPF][WPT];
    float4 sr[CPF];  // group scales of this lane's row for a chunk's 4 groups
    auto load_chunk = [&](int c, int j) {
        const int k0 = kb + c * KC;
#pragma unroll
        for (int u = 0; u < XPT; ++u) {
            const int i = tid + u * kThreads;
            if (i < XV) {
                const int r = i / (KC / 4), c4 = i % (KC / 4);
                const int m = min(m0 + r, M - 1);
                xr[j][u] = *reinterpret_cast<const float4*>(x + (size_t)m * ldx + k0 + c4 * 4);
                if constexpr (NORM) {
                    gr[j][u] = *reinterpret_cast<const float4*>(nw + k0 + c4 * 4);
                    rr[j][u] = DEFER ? 1.0f : rs[m];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < WPT; ++u) {
            const int i = tid + u * kThreads;
            if (i < WV) {
                const int r = i / (KC / 16), c16 = i % (KC / 16);
                const int n = min(n0 + r, NR - 1);
                if constexpr (TL)
                    wr[j][u] = *reinterpret_cast<const int4*>(q + tm_off(tmap, n, k0 + c16 * 16));
                else
                    wr[j][u] = *reinterpret_cast<const int4*>(q + (size_t)n * K + k0 + c16 * 16);
            }
        }
        if constexpr (!ROWSCALE) {
            if constexpr (TL) {
                const int g0 = k0 >> 5;
                sr[j] = make_float4(sc[tm_scale(tmap, nrow, g0)], sc[tm_scale(tmap, nrow, g0 + 1)],
                                    sc[tm_scale(tmap, nrow, g0 + 2)],
                                    sc[tm_scale(tmap, nrow, g0 + 3)]);
            } else {
                sr[j] = *reinterpret_cast<const float4*>(sc + (size_t)nrow * nblk + (k0 >> 5));
            }
        }
    };
    auto store_chunk = [&](int j) {
#pragma unroll
        for (int u = 0; u < XPT; ++u) {
            const int i = tid + u * kThreads;
            if (i < XV) {
                const int r = i / (KC / 4), c4 = i % (KC / 4);
                float4 v = xr[j][u];
                if constexpr (NORM) v = norm4(v, rr[j][u], gr[j][u]);
                store_hilo(&xs_hi[r * XP + c4 * 4], &xs_lo[r * XP + c4 * 4], v);
            }
        }
#pragma unroll
        for (int u = 0; u < WPT; ++u) {
            const int i = tid + u * kThreads;
            if (i < WV) {
                const int r = i / (KC / 16), c16 = i % (KC / 16);
                store_w16(&ws[r * WP + c16 * 16], wr[j][u]);
            }
        }
    };

    f32x4 acc[TM];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) acc[tm] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int nch = kper / KC;
#pragma unroll
    for (int j = 0; j < CPF; ++j)
        if (j < nch) load_chunk(j, j);
    for (int c0 = 0; c0 < nch; c0 += CPF)
#pragma unroll
    for (int j = 0; j < CPF; ++j) {
        const int c = c0 + j;
        if (c >= nch) break;  // uniform
        const float4 s_cur = sr[j];
        __syncthreads();
        store_chunk(j);
        __syncthreads();
        if (c + CPF < nch) load_chunk(c + CPF, j);
        const float sg[4] = {s_cur.x, s_cur.y, s_cur.z, s_cur.w};
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int kofs = g * 32 + (lane >> 4) * 8;
            const bf16x8 bw = *reinterpret_cast<const bf16x8*>(&ws[(wave * 16 + (lane & 15)) * WP + kofs]);
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) {
                const int r = tm * 16 + (lane & 15);
                const bf16x8 ah = *reinterpret_cast<const bf16x8*>(&xs_hi[r * XP + kofs]);
                const bf16x8 al = *reinterpret_cast<const bf16x8*>(&xs_lo[r * XP + kofs]);
                if constexpr (ROWSCALE) {
                    acc[tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bw, acc[tm], 0, 0, 0);
                    acc[tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bw, acc[tm], 0, 0, 0);
                } else {
                    f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bw, d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bw, d, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[tm][i] = fmaf(d[i], sg[g], acc[tm][i]);
                }
            }
        }
    }
    if constexpr (ROWSCALE) {
        const float s = sc[nrow];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[tm][i] *= s;
    }
    if (ncol < NR) {
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + tm * 16 + (lane >> 4) * 4 + i;
                if (m < M) part[((size_t)ks * M + m) * ldp + ncol] = acc[tm][i];
            }
    }
}


// RMSNorm row scales rs[m] = 1/sqrt(mean(x[m]^2) + eps): every load of the
// row is issued before the sum (K <= 4096 per pass of 256 x float4).
__global__ __launch_bounds__(kThreads) void k_row_rs(const float* __restrict__ x, int ldx, int K,
                                                     float eps, float* __restrict__ rs) {
    __shared__ float red[kThreads / QLM_WAVE];
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)blockIdx.x * ldx);
    const int n4 = K >> 2;
    float ss = 0.0f;
    for (int b = 0; b < n4; b += 4 * kThreads) {
        float4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = b + u * kThreads + threadIdx.x;
            v[u] = i < n4 ? xr[i] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ss = fmaf(v[u].x, v[u].x, ss);
            ss = fmaf(v[u].y, v[u].y, ss);
            ss = fmaf(v[u].z, v[u].z, ss);
            ss = fmaf(v[u].w, v[u].w, ss);
        }
    }
    ss = block_sum(ss, red);
    if (threadIdx.x == 0) rs[blockIdx.x] = 1.0f / sqrtf(ss / (float)K + eps);
}

// The activation of the many-row matmul split once into bf16 hi and lo planes
// (the lo plane M * K after the hi one), with the RMSNorm applied when NORM.
// A plane holds 32-row tiles (the last one of M % 32 rows) as [octet of
// columns][row][8]: k_mm_pf's workgroups copy it to LDS as it is, 1 KB
// contiguous a wave and load. A workgroup takes kSplitRows rows and the
// octets blockIdx.y * per .. + per - 1 of them; the row sums of NORM are its own (32
// lanes a row), which spares a launch of their own.
constexpr int kSplitRows = 8;

template <bool NORM>
__global__ __launch_bounds__(kThreads) void k_split_op(const float* __restrict__ x, int ldx,
                                                      const float* __restrict__ nw, float eps,
                                                      int M, int K, int per,
                                                      uint16_t* __restrict__ xs) {
    __shared__ float srs[kSplitRows];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.x * kSplitRows;
    if constexpr (NORM) {
        const int m = min(m0 + (tid >> 5), M - 1);
        const float4* xr = reinterpret_cast<const float4*>(x + (size_t)m * ldx);
        const int n4 = K >> 2;
        float ss = 0.0f;
        for (int b = tid & 31; b < n4; b += 32 * 8) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = xr[min(b + 32 * u, n4 - 1)];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float4 e = b + 32 * u < n4 ? v[u] : make_float4(0.f, 0.f, 0.f, 0.f);
                ss = fmaf(e.x, e.x, ss);
                ss = fmaf(e.y, e.y, ss);
                ss = fmaf(e.z, e.z, ss);
                ss = fmaf(e.w, e.w, ss);
            }
        }
        ss = group_sum<32>(ss);
        if ((tid & 31) == 0) srs[tid >> 5] = 1.0f / sqrtf(ss / (float)K + eps);
        __syncthreads();
    }
    const int r = tid & (kSplitRows - 1), m = m0 + r;
    if (m >= M) return;
    const int T = m >> 5, R = min(32, M - 32 * T);
    const float s = NORM ? srs[r] : 1.0f;
    const float* xr = x + (size_t)m * ldx;
    uint16_t* dst = xs + (size_t)T * 32 * K + (m & 31) * 8;
    const int o1 = min(K >> 3, (int)(blockIdx.y + 1) * per);
#pragma unroll 2
    for (int o = blockIdx.y * per + tid / kSplitRows; o < o1; o += kThreads / kSplitRows) {
        float4 v[2];
        v[0] = *reinterpret_cast<const float4*>(xr + o * 8);
        v[1] = *reinterpret_cast<const float4*>(xr + o * 8 + 4);
        if constexpr (NORM) {
            v[0] = norm4(v[0], s, *reinterpret_cast<const float4*>(nw + o * 8));
            v[1] = norm4(v[1], s, *reinterpret_cast<const float4*>(nw + o * 8 + 4));
        }
        uint16_t* d = dst + (size_t)o * R * 8;
        __attribute__((aligned(16))) unsigned short h[8], l[8];
        store_hilo(h, l, v[0]);
        store_hilo(h + 4, l + 4, v[1]);
        *reinterpret_cast<uint4*>(d) = *reinterpret_cast<const uint4*>(h);
        *reinterpret_cast<uint4*>(d + (size_t)M * K) = *reinterpret_cast<const uint4*>(l);
    }
}

// 128 octets (1024 columns) a workgroup: enough workgroups for a few rows
int launch_split(const float* x, int ldx, const float* nw, float eps, int M, int K, uint16_t* xs,
                 hipStream_t st) {
    constexpr int kPer = 128;
    const dim3 grid((M + kSplitRows - 1) / kSplitRows, ((K >> 3) + kPer - 1) / kPer);
    if (nw)
        hipLaunchKernelGGL(k_split_op<true>, grid, dim3(kThreads), 0, st, x, ldx, nw, eps, M, K,
                           kPer, xs);
    else
        hipLaunchKernelGGL(k_split_op<false>, grid, dim3(kThreads), 0, st, x, ldx, nw, eps, M, K,
                           kPer, xs);
    return qlm_launch_status();
}

// K slices for the M <= 64 path: the fewest that divide the 128-column
// chunk count and give each workgroup at most 6 chunks and the launch at
// least ~640 workgroups (up to 16 rows); above 16 rows (four times the work
// a workgroup) at most 8 chunks a workgroup, ~320 workgroups and at least 8
// slices. A tall matrix (>= 1024 row tiles) is one slice. Measured on the
// config-1 shapes (graph replays): 4096 x 12288 at 4 / 16 rows 21.4 / 23.1
// us with the former rule (at most 4 chunks a workgroup) against 18.2 /
// 20.4 us; 64 rows 40.9 against 38.5 us; 4096 x 4096 at 64 rows 22.4
// against 20.7 us; 12288 x 4096 at 64 rows 42.6 us in 8 slices, 43.1 in 4.
int sk_splits(int M, int NR, int K) {
    const int nt = (NR + kSkRows - 1) / kSkRows;
    const int nch = K / kSkKc;
    if (nt >= 1024) return 1;
    const bool tall = M > 16;
    const int per = tall ? 8 : 6;
    const int wgs = tall ? 320 : 640;
    int want = (nch + per - 1) / per;
    want = want > (wgs + nt - 1) / nt ? want : (wgs + nt - 1) / nt;
    if (tall && want < 8) want = 8;
    for (int d = 1; d <= nch; ++d)
        if (nch % d == 0 && d >= want) return d;
    return nch;
}

bool use_sk(int M, int K) { return M <= 64 && K % kSkKc == 0; }

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace
extern "C" size_t qlm_matmul_i8_rows64_workspace_bytes(int M, int N, int K, int epilogue);
extern "C" int qlm_matmul_i8_rows64(const float* x, int ldx, const float* norm_w, float eps,
                                    const int8_t* q_tiles, const float* s_rows, float* y,
                                    int ldy, int M, int N, int K, int epilogue, void* work,
                                    size_t work_bytes, void* stream);
namespace {

// the tile-major 2..64-row form with one scale per weight row (gemm_mx.hip),
// where measured faster than the K-sliced bf16 form: N >= 8192 (32 or more
// 256-row tile groups), or more than 16 rows and K > 4096. With fewer groups
// its K slices and their reduction launch cost more (4096 x 4096: 15.4
// against 12.6 us at 16 rows, 27.5 against 23.3 us at 64)
bool rows64_applies(int M, int N, int K, int group, int epi) {
    if (N < 8192 && (M <= 16 || K <= 4096)) return false;
    return group == K && M >= 2 && M <= 64 && K % 64 == 0 && epi != EPI_SWIGLU;
}

// the split activation (bf16 hi, lo), the least a many-row launch needs
size_t pf_base_bytes(int M, int K) {
    return align256((size_t)M * sizeof(float)) + align256((size_t)4 * M * K);
}

// with room for the slices of any such launch of up to M rows (at most
// kPfBlocks workgroups' sums, and no more rows than there are)
size_t pf_workspace(int M, int K) {
    return pf_base_bytes(M, K) + (size_t)kPfBlocks * kPfN * sizeof(float) * (M < kPfM ? M : kPfM);
}

// full: what a launch can use; otherwise the least it accepts (a many-row
// launch then takes the K slices that fit)
size_t mm_workspace(int M, int N, int K, int epi, bool full) {
    size_t b = align256((size_t)M * sizeof(float));  // row scales
    if (use_sk(M, K)) {
        const int NR = epi == EPI_SWIGLU ? 2 * N : N;
        const int ks = sk_splits(M, NR, K);
        if (!(ks == 1 && epi == EPI_STORE)) b += (size_t)ks * M * NR * sizeof(float);
    } else {
        b = full ? pf_workspace(M, K) : pf_base_bytes(M, K);
    }
    // room for the 2..64-row digit form of qlm_matmul_i8_tm (one scale per
    // weight row); the query cannot tell which scales a caller holds
    if (M >= 2 && M <= 64 && K % 64 == 0 && epi != EPI_SWIGLU) {
        const size_t r = qlm_matmul_i8_rows64_workspace_bytes(M, N, K, epi);
        if (r > b) b = r;
    }
    return b;
}

template <int TM, bool RS, bool NORM, bool DEFER, bool TL>
void launch_sk(const float* x, int ldx, const float* rs, const float* nw, const int8_t* q,
               const float* sc, float* part, int ldp, int M, int NR, int K, int ks,
               const TileMap& tm, hipStream_t st) {
    const dim3 grid((NR + kSkRows - 1) / kSkRows, ks, (M + 16 * TM - 1) / (16 * TM));
    hipLaunchKernelGGL((k_mm_i8_sk<TM, RS, NORM, DEFER, TL>), grid, dim3(kThreads), 0, st, x, ldx,
                       rs, nw, q, sc, part, ldp, M, NR, K, K / ks, tm);
}

template <bool RS, bool NORM, bool DEFER, bool TL>
void launch_sk_tm(const float* x, int ldx, const float* rs, const float* nw, const int8_t* q,
                  const float* sc, float* part, int ldp, int M, int NR, int K, int ks,
                  const TileMap& tm, hipStream_t st) {
    if (M <= 16)
        launch_sk<1, RS, NORM, DEFER, TL>(x, ldx, rs, nw, q, sc, part, ldp, M, NR, K, ks, tm, st);
    else if (M <= 32)
        launch_sk<2, RS, NORM, DEFER, TL>(x, ldx, rs, nw, q, sc, part, ldp, M, NR, K, ks, tm, st);
    else
        launch_sk<4, RS, NORM, DEFER, TL>(x, ldx, rs, nw, q, sc, part, ldp, M, NR, K, ks, tm, st);
}

template <int EPI, bool NORM>
void launch_reduce(const float* part, int ks, int M, int NR, int N, float* y, int ldy,
                   const float* x, int ldx, int K, float eps, hipStream_t st) {
    const dim3 grid((N + kThreads - 1) / kThreads, M);
    hipLaunchKernelGGL((k_mm_reduce<EPI, NORM>), grid, dim3(kThreads), 0, st, part, ks, M, NR, N,
                       y, ldy, x, ldx, K, eps);
}

// K slices of a many-row launch: the count with the least modelled time. A
// workgroup alone on its CU takes about 1.0 us a 32-column group (without
// group scales 0.78), two together 1.65 (1.41) for both; slices cost a reduction
// launch and their sums' way through memory, 8 us + 0.45 us a MB. Measured
// (one slice -> chosen): down projection 2560 x 9728 at 65 / 511 / 2048 rows
// 283 -> 36 / 290 -> 75 / 309 -> 248 us; in-projection 8224 x 2560 at 128
// rows 84 -> 37 us; gate/up stays whole from 300 rows (91 us; 103 in two).
int pf_splits(int M, int N, int K, int epi, bool chained) {
    const int bn = epi == EPI_SWIGLU ? kPfN / 2 : kPfN;
    const long tiles = (long)((N + bn - 1) / bn) * ((M + kPfM - 1) / kPfM);
    const double t1 = chained ? 0.78 : 1.0, t2 = chained ? 1.41 : 1.65;
    const double mb = (double)M * (epi == EPI_SWIGLU ? 2.0 * N : N) * 4e-6;
    const int ngrp = K / 32;
    int best = 1;
    double least = 0.0;
    for (int ks = 1; ks <= 16 && (ks == 1 || (tiles * ks <= kPfBlocks && ngrp >= 4 * ks)); ++ks) {
        const long c = (tiles * ks + 255) / 256;
        const double t = ((double)(c / 2) * t2 + (double)(c & 1) * t1) * ((ngrp + ks - 1) / ks) +
                         (ks > 1 ? 8.0 + 0.45 * mb * ks : 0.0);
        if (ks == 1 || t < least) {
            least = t;
            best = ks;
        }
    }
    return best;
}

size_t pf_part_bytes(int ks, int M, int N, int epi) {
    return ks > 1 ? (size_t)ks * M * (epi == EPI_SWIGLU ? 2 * N : N) * sizeof(float) : 0;
}

template <int WK, bool RS, int EPI>
int launch_pf_e(PfArgs a, int ks, hipStream_t st) {
    const dim3 grid(8 * ((a.blocks + 7) / 8));
    if (ks > 1)
        hipLaunchKernelGGL((k_mm_pf<WK, RS, EPI, true>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((k_mm_pf<WK, RS, EPI, false>), grid, dim3(256), 0, st, a);
    return qlm_launch_status();
}

// Many rows: the activation split (RMSNorm applied), the matmul, and the
// ordered sum of its K slices where there are several. `work` holds the split
// activation and then the slices' sums.
template <int WK, bool RS>
int pf_run(const float* x, int ldx, const float* nw, float eps, const void* q, const float* sc,
           float* y, int ldy, int M, int N, int K, int epi, void* work, size_t work_bytes,
           hipStream_t st) {
    uint16_t* xs = static_cast<uint16_t*>(work);
    int rc = launch_split(x, ldx, nw, eps, M, K, xs, st);
    if (rc != QLM_OK) return rc;
    const size_t xsb = align256((size_t)4 * M * K);
    float* part = reinterpret_cast<float*>(static_cast<char*>(work) + xsb);
    const int NR = epi == EPI_SWIGLU ? 2 * N : N;
    int ks = pf_splits(M, N, K, epi, RS || WK == W_BF16);
    while (ks > 1 && xsb + pf_part_bytes(ks, M, N, epi) > work_bytes) --ks;
    const int bn = epi == EPI_SWIGLU ? kPfN / 2 : kPfN;
    const int ngrp = K / 32;
    PfArgs a{xs, q, sc, ks > 1 ? part : y, ldy, M, N, K, (N + bn - 1) / bn,
             (M + kPfM - 1) / kPfM, 0, (ngrp + ks - 1) / ks};
    ks = (ngrp + a.gslice - 1) / a.gslice;  // no empty slice
    a.blocks = a.gx * a.gy * ks;
    if (epi == EPI_SWIGLU)
        rc = launch_pf_e<WK, RS, EPI_SWIGLU>(a, ks, st);
    else if (epi == EPI_RESID && ks == 1)
        rc = launch_pf_e<WK, RS, EPI_RESID>(a, ks, st);
    else
        rc = launch_pf_e<WK, RS, EPI_STORE>(a, ks, st);
    if (rc != QLM_OK || ks == 1) return rc;
    if (epi == EPI_SWIGLU)
        launch_reduce<EPI_SWIGLU, false>(part, ks, M, NR, N, y, ldy, x, ldx, K, eps, st);
    else if (epi == EPI_RESID)
        launch_reduce<EPI_RESID, false>(part, ks, M, NR, N, y, ldy, x, ldx, K, eps, st);
    else
        launch_reduce<EPI_STORE, false>(part, ks, M, NR, N, y, ldy, x, ldx, K, eps, st);
    return qlm_launch_status();
}

template <int EPI, bool NORM>
int launch_mm16(const float* x, int ldx, const float* rs, const float* nw, const uint16_t* w,
                float* y, int ldy, int M, int N, int K, hipStream_t st) {
    constexpr int BN_OUT = EPI == EPI_SWIGLU ? 64 : 128;
    const dim3 grid((N + BN_OUT - 1) / BN_OUT, (M + 127) / 128);
    if (K % 64 == 0)
        hipLaunchKernelGGL((k_mm_bf16<EPI, NORM, 2>), grid, dim3(kThreads), 0, st, x, ldx, rs, nw,
                           w, y, ldy, M, N, K);
    else
        hipLaunchKernelGGL((k_mm_bf16<EPI, NORM, 1>), grid, dim3(kThreads), 0, st, x, ldx, rs, nw,
                           w, y, ldy, M, N, K);
    return qlm_launch_status();
}

template <bool RS, bool NORM, bool TL>
int mm_run(const float* x, int ldx, float* rs, const float* nw, float eps, const int8_t* q,
           const float* sc, float* y, int ldy, int M, int N, int K, int epi, float* part,
           size_t work_bytes, hipStream_t st) {
    const TileMap tm{N, (N + 15) / 16, K / 64};  // a SwiGLU matrix: gate rows, then up rows
    if (use_sk(M, K)) {
        const int NR = epi == EPI_SWIGLU ? 2 * N : N;
        const int ks = sk_splits(M, NR, K);
        const bool direct = ks == 1 && epi == EPI_STORE;
        float* dst = direct ? y : part;
        const int ldp = direct ? ldy : NR;
        if (direct) {  // the matmul writes y itself: row scales first
            if constexpr (NORM) {
                hipLaunchKernelGGL(k_row_rs, dim3(M), dim3(kThreads), 0, st, x, ldx, K, eps, rs);
                const int rc = qlm_launch_status();
                if (rc != QLM_OK) return rc;
            }
            launch_sk_tm<RS, NORM, false, TL>(x, ldx, rs, nw, q, sc, dst, ldp, M, NR, K, ks, tm,
                                              st);
            return qlm_launch_status();
        }
        // row scales folded into the reduction (no separate launch)
        launch_sk_tm<RS, NORM, NORM, TL>(x, ldx, rs, nw, q, sc, dst, ldp, M, NR, K, ks, tm, st);
        int rc = qlm_launch_status();
        if (rc != QLM_OK) return rc;
        if (epi == EPI_STORE)
            launch_reduce<EPI_STORE, NORM>(part, ks, M, NR, N, y, ldy, x, ldx, K, eps, st);
        else if (epi == EPI_RESID)
            launch_reduce<EPI_RESID, false>(part, ks, M, NR, N, y, ldy, x, ldx, K, eps, st);
        else
            launch_reduce<EPI_SWIGLU, NORM>(part, ks, M, NR, N, y, ldy, x, ldx, K, eps, st);
        return qlm_launch_status();
    }
    return pf_run<TL ? W_TILES : W_ROWS, RS>(x, ldx, NORM ? nw : nullptr, eps, q, sc, y, ldy, M, N,
                                             K, epi, rs, work_bytes, st);
}

}  // namespace

extern "C" size_t qlm_matmul_i8_workspace_bytes(int M, int N, int K, int epilogue) {
    if (M <= 0 || N <= 0 || K <= 0 || epilogue < EPI_STORE || epilogue > EPI_SWIGLU) return 0;
    // 16 and 64 rows are the last of a K-slice rule and can need more than the
    // rows after them (64: 50 MB, 65: 35 MB for a gate/up of 2 x 9728 x 2560)
    size_t b = mm_workspace(M, N, K, epilogue, true);
    for (const int m : {16, 64})
        if (m < M) b = std::max(b, mm_workspace(m, N, K, epilogue, true));
    return b;
}

extern "C" size_t qlm_matmul_bf16_workspace_bytes(int M, int K) {
    if (M <= 0 || K <= 0) return 0;
    return pf_workspace(M, K);
}

extern "C" int qlm_matmul_bf16(const float* x, int ldx, const float* norm_w, float eps,
                               const uint16_t* w, float* y, int ldy, int M, int N, int K,
                               int epilogue, void* work, size_t work_bytes, void* stream) {
    if (!x || !w || !y || M <= 0 || N <= 0 || K <= 0) return QLM_ERR_ARG;
    if (epilogue < EPI_STORE || epilogue > EPI_SWIGLU) return QLM_ERR_ARG;
    if (epilogue == EPI_SWIGLU && !norm_w) return QLM_ERR_ARG;
    if (epilogue == EPI_RESID && norm_w) return QLM_ERR_ARG;
    if (K % 32 != 0 || ldx < K || ldx % 4 != 0 || ldy < N) return QLM_ERR_SHAPE;
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_w | (uintptr_t)work) & 15u)
        return QLM_ERR_SHAPE;
    hipStream_t st = as_stream(stream);
    if (norm_w && (!work || work_bytes < align256((size_t)M * sizeof(float)))) return QLM_ERR_ARG;
    if (work && work_bytes >= pf_base_bytes(M, K))
        return pf_run<W_BF16, false>(x, ldx, norm_w, eps, w, nullptr, y, ldy, M, N, K, epilogue,
                                     work, work_bytes, st);
    float* rs = static_cast<float*>(work);
    if (norm_w) {
        hipLaunchKernelGGL(k_row_rs, dim3(M), dim3(kThreads), 0, st, x, ldx, K, eps, rs);
        const int rc = qlm_launch_status();
        if (rc != QLM_OK) return rc;
    }
    // a smaller workspace: each workgroup converts its activation chunks itself
    if (epilogue == EPI_SWIGLU)
        return launch_mm16<EPI_SWIGLU, true>(x, ldx, rs, norm_w, w, y, ldy, M, N, K, st);
    if (epilogue == EPI_RESID)
        return launch_mm16<EPI_RESID, false>(x, ldx, nullptr, nullptr, w, y, ldy, M, N, K,
                                                    st);
    if (norm_w)
        return launch_mm16<EPI_STORE, true>(x, ldx, rs, norm_w, w, y, ldy, M, N, K, st);
    return launch_mm16<EPI_STORE, false>(x, ldx, nullptr, nullptr, w, y, ldy, M, N, K, st);
}

namespace {
template <bool TL>
int matmul_i8_entry(const float* x, int ldx, const float* norm_w, float eps, const int8_t* q,
                    const float* scales, int group, float* y, int ldy, int M, int N, int K,
                    int epilogue, void* work, size_t work_bytes, void* stream) {
    if (!x || !q || !scales || !y) return QLM_ERR_ARG;
    if (M <= 0 || N <= 0 || K <= 0) return QLM_ERR_ARG;
    if (epilogue < EPI_STORE || epilogue > EPI_SWIGLU) return QLM_ERR_ARG;
    if (K % (TL ? 64 : 32) != 0) return QLM_ERR_SHAPE;
    const bool rowscale = (group == K);
    if (!rowscale && group != 32) return QLM_ERR_SHAPE;
    if (ldx < K || ldy < N || ldx % 4 != 0) return QLM_ERR_SHAPE;
    if (((uintptr_t)x | (uintptr_t)q | (uintptr_t)norm_w | (uintptr_t)scales) & 15u)
        return QLM_ERR_SHAPE;
    const size_t need = mm_workspace(M, N, K, epilogue, false);
    if (!work || work_bytes < need || ((uintptr_t)work & 15u)) return QLM_ERR_ARG;
    if constexpr (TL) {
        // 2..64 rows with one scale per weight row: int8 digits on the int8
        // matrix cores (its workspace needs 256-byte alignment)
        if (rows64_applies(M, N, K, group, epilogue) && !(epilogue == EPI_RESID && norm_w) &&
            ((uintptr_t)work & 255u) == 0) {
            const int rc = qlm_matmul_i8_rows64(x, ldx, norm_w, eps, q, scales, y, ldy, M, N, K,
                                                epilogue, work, work_bytes, stream);
            if (rc != QLM_ERR_SHAPE) return rc;
        }
    }
    hipStream_t st = as_stream(stream);
    float* rs = reinterpret_cast<float*>(work);
    float* part = reinterpret_cast<float*>(reinterpret_cast<char*>(work) + align256((size_t)M * 4));
    if (norm_w)
        return rowscale ? mm_run<true, true, TL>(x, ldx, rs, norm_w, eps, q, scales, y, ldy, M, N,
                                                 K, epilogue, part, work_bytes, st)
                        : mm_run<false, true, TL>(x, ldx, rs, norm_w, eps, q, scales, y, ldy, M,
                                                  N, K, epilogue, part, work_bytes, st);
    return rowscale ? mm_run<true, false, TL>(x, ldx, rs, nullptr, eps, q, scales, y, ldy, M, N, K,
                                              epilogue, part, work_bytes, st)
                    : mm_run<false, false, TL>(x, ldx, rs, nullptr, eps, q, scales, y, ldy, M, N,
                                               K, epilogue, part, work_bytes, st);
}
}  // namespace

extern "C" int qlm_matmul_i8(const float* x, int ldx, const float* norm_w, float eps,
                             const int8_t* q, const float* scales, int group, float* y, int ldy,
                             int M, int N, int K, int epilogue, void* work, size_t work_bytes,
                             void* stream) {
    return matmul_i8_entry<false>(x, ldx, norm_w, eps, q, scales, group, y, ldy, M, N, K,
                                  epilogue, work, work_bytes, stream);
}

extern "C" int qlm_matmul_i8_tm(const float* x, int ldx, const float* norm_w, float eps,
                                const int8_t* q_tiles, const float* s_tiles, int group, float* y,
                                int ldy, int M, int N, int K, int epilogue, void* work,
                                size_t work_bytes, void* stream) {
    return matmul_i8_entry<true>(x, ldx, norm_w, eps, q_tiles, s_tiles, group, y, ldy, M, N, K,
                                 epilogue, work, work_bytes, stream);
}

// Loads this file's code object on the current device now; the runtime
// otherwise loads it at the first launch of one of its kernels (4-20 ms,
// measured inside a first prefill or decode step).
hipError_t qlm_load_gemm() {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(k_row_rs));
}
