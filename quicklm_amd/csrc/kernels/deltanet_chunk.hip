// Chunked prefill of a Gated DeltaNet layer (one sequence, T prompt rows at
// positions p0 .. p0+T-1). The reference runs the recurrence row by row
// (Qwen3_5GatedDeltaNet::forward_chunk, attention.cpp:600-758); this is the
// same recurrence in the chunked "WY" form, with every contraction on the
// fp32 matrix cores (v_mfma_f32_16x16x4f32).
//
// Per head, with the state S [d_k, d_v] before a chunk of C = 64 rows,
// alpha_t = log-decay, G_t = sum_{s<=t} alpha_s within the chunk,
// gamma_t = exp(G_t), beta_t the write strength and q, k L2-normalised:
//   S_t = gamma_t S + sum_{s<=t} (gamma_t/gamma_s) k_s w_s^T, where
//   (I + A) W = diag(beta) (V - diag(gamma) K S),
//   A[t][s] = beta_t (gamma_t/gamma_s) (k_t . k_s) for s < t.
// With T = (I + A)^-1 diag(beta): U = T V, Wk = T diag(gamma) K, W = U - Wk S,
//   o_t = (gamma_t (Q S)[t] + sum_{s<=t} (gamma_t/gamma_s)(q_t . k_s) w_s) / sqrt(d),
//   S_next = gamma_end S + K^T diag(gamma_end/gamma) W.
// Every decay factor is exp of a non-positive number (ratios, never 1/gamma).
//
// Kernels (one stream, in order):
//   k_dn_chunk_prep   per (8 or 16 rows, head): conv taps from the prompt rows or
//                     the ring (positions before p0), SiLU, L2 norms, gates --
//                     the decode step's arithmetic;
//   k_dn_chunk_intra  per (chunk, head): everything that does not depend on
//                     the state: the masked, decayed K K^T and Q K^T, the
//                     inverse (I + A)^-1 by blocks of 16, U, Wk and the decayed
//                     K^T;
//   k_dn_chunk_chain  per (head, 16 value columns): chunks in order, W and the
//                     state only;
//   k_dn_chunk_out    per (chunk, head): the outputs from the states and W of
//                     all chunks at once, head RMSNorm + SiLU(z) gate (decode
//                     arithmetic) and the conv ring rows of the last positions.
//
// Operand order. A 16x16 block feeds or leaves a matrix instruction as one
// float4 a lane: lane (l16, l4) holds its elements (l16, 4 l4 .. + 3), rows
// first as the A operand and columns first as the B operand, where the K
// index of product j of a block is 4 l4 + j; a result D holds (rows 4 l4 + i,
// column l16), which is the B operand's order of the same matrix and the A
// operand's of its transpose. So every matrix that one kernel hands to the
// next is stored block by block, 1 KB each, lane after lane, and a product's
// result is the next product's operand without a transposition.

#include "common.hpp"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kD = 128;      // head dim (d_k = d_v)
constexpr int kC = 64;       // chunk rows
constexpr int KP = kD + 4;   // padded LDS row of a [64][128] tile
constexpr int TP = kC + 4;   // padded LDS row of a [64][64] tile
constexpr int CB = 16;       // value columns per chain workgroup
constexpr int kBlk = 256;    // floats of a 16x16 block in operand order

// D += A B on a 16x16 tile, K = 4: lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; it holds D[(l/16)*4 + i][l%16].
__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Four products of one block pair: K = 16.
__device__ __forceinline__ f32x4 mma4(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = mma(a[j], b[j], c);
    return c;
}

__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }

// q, k, v and gate rows are kept by chunk and head: row t of head h is row
// t % kC of tile (t / kC, h).
__device__ __forceinline__ size_t gix(int t, int h, int H) {
    return ((size_t)(t / kC) * H + h) * kC + t % kC;
}
__device__ __forceinline__ size_t rix(int t, int h, int H) { return gix(t, h, H) * kD; }

// Per (PR rows, head): thread (section, column) slides the conv window down
// the rows, the q and k outputs wait in LDS for their row norms (6 waves, a
// norm each at a time), v goes straight out. 16 heads, us at 4 / 8 / 16 / 32
// rows a workgroup: 66 rows 5.0 / 5.0 / 7.7 / 12.4, 300 rows 9.2 / 8.9 / 10.9 /
// 12.9, 700 rows 16.6 / 14.6 / 14.7 / 19.9, 2047 rows 38.6 / 32.2 / 32.0 / 33.2
// (there bound by the vector work of the SiLUs and divisions as much as by its
// 100 MB): 8 rows while the workgroups are few, 16 above.
template <int PR>
__global__ __launch_bounds__(3 * kD) void k_dn_chunk_prep(
    const float* __restrict__ proj, int ldp, int T, const float* __restrict__ conv_state,
    const float* __restrict__ wt, const float* __restrict__ A_log,
    const float* __restrict__ dt_bias, int p0, int H, float* __restrict__ qn,
    float* __restrict__ kn, float* __restrict__ vv, float* __restrict__ alpha,
    float* __restrict__ beta) {
    __shared__ float ys[2][PR][kD];
    const int t0 = blockIdx.x * PR, h = blockIdx.y, tid = threadIdx.x;
    const int nt = min(PR, T - t0);
    const int lane = tid & 63, wave = tid >> 6;
    const int HD = H * kD, C = 3 * HD;
    const int sec = tid / kD, tt = tid % kD, ch = sec * HD + h * kD + tt;
    const float w0 = wt[ch], w1 = wt[(size_t)C + ch], w2 = wt[(size_t)2 * C + ch],
                w3 = wt[(size_t)3 * C + ch];
    // inputs of positions t-3, t-2, t-1; positions before p0 come from the
    // ring, row (position mod 3), as the decode step reads it (zero rows on a
    // fresh sequence)
    float xw[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int r = t0 - 3 + j;
        if (r >= 0) {
            xw[j] = proj[(size_t)r * ldp + ch];
        } else {
            const int row = ((p0 + r) % 3 + 3) % 3;
            xw[j] = conv_state[(size_t)row * C + ch];
        }
    }
    float xr[PR];  // rows past T read row T-1 and are never stored
#pragma unroll
    for (int r = 0; r < PR; ++r) xr[r] = proj[(size_t)min(t0 + r, T - 1) * ldp + ch];
#pragma unroll
    for (int r = 0; r < PR; ++r) {
        float acc = 0.0f;
        acc = nc_add_mul(acc, xw[0], w0);
        acc = nc_add_mul(acc, xw[1], w1);
        acc = nc_add_mul(acc, xw[2], w2);
        acc = nc_add_mul(acc, xr[r], w3);
        const float y = silu_f(acc);
        if (sec < 2) ys[sec][r][tt] = y;
        else if (r < nt) vv[rix(t0 + r, h, H) + tt] = y;
        xw[0] = xw[1];
        xw[1] = xw[2];
        xw[2] = xr[r];
    }
    if (tid >= 2 * kD && tid - 2 * kD < nt) {
        const int t = t0 + tid - 2 * kD;
        const float* pr = proj + (size_t)t * ldp;
        const float dt = pr[4 * HD + H + h] + dt_bias[h];
        const float sp = dt > 20.0f ? dt : log1pf(expf(dt));
        alpha[gix(t, h, H)] = -expf(A_log[h]) * sp;
        beta[gix(t, h, H)] = 1.0f / (1.0f + expf(-pr[4 * HD + h]));
    }
    __syncthreads();
    for (int i = wave; i < 2 * PR; i += 3 * kD / 64) {
        const int which = i & 1, r = i >> 1;
        if (r >= nt) break;
        const float a0 = ys[which][r][lane], a1 = ys[which][r][lane + 64];
        float ss = fmaf(a0, a0, a1 * a1);
        ss = wave_sum(ss);
        const float nrm = sqrtf(ss + 1e-6f);
        float* dst = (which == 0 ? qn : kn) + rix(t0 + r, h, H);
        dst[lane] = a0 / nrm;
        dst[lane + 64] = a1 / nrm;
    }
}

// What a chunk's state-independent part is bound by is the fp32 matrix cores
// and the latency of its steps in turn, at two workgroups a CU. The products
// above the diagonal are left out (K K^T, Q K^T, U and Wk: 10 of 16 blocks),
// and the inverse goes by blocks: each wave inverts one diagonal block (a
// column a lane, 16 steps), then
//   [X0 0; -X1 L X0, X1] joins blocks to 32 and to 64 rows,
// whose two products chain in registers. kk: the chunk's k rows in, the
// decayed K^T out (all rows are in LDS before the first is overwritten).
__global__ __launch_bounds__(256, 2) void k_dn_chunk_intra(
    const float* __restrict__ qn, float* kk, const float* __restrict__ vv,
    const float* __restrict__ alpha, const float* __restrict__ beta, int T, int H,
    float* __restrict__ U, float* __restrict__ Wk, float* __restrict__ Mq,
    float* __restrict__ Gc) {
    __shared__ __attribute__((aligned(16))) float Ks[kC * KP];
    __shared__ __attribute__((aligned(16))) float Ts[kC * TP];  // A
    __shared__ __attribute__((aligned(16))) float Xs[kC * TP];  // (I + A)^-1
    __shared__ __attribute__((aligned(16))) float gs[kC], bs[kC], bg[kC], dec[kC];
    const int c = blockIdx.x, h = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    const int nt = min(kC, T - c * kC);
    const size_t tile = (size_t)c * H + h;
    const size_t base = tile * kC * kD;

    // operands of later products that come straight from memory, requested
    // first: q rows of this wave's row block, v's 32 columns of this wave
    // (rows past the last are read as the last and masked at use)
    const int tq = wave * 16 + l16;
    f32x4 qv[kD / 16];
#pragma unroll
    for (int kb = 0; kb < kD / 16; ++kb)
        qv[kb] = ld4(qn + base + (size_t)min(tq, nt - 1) * kD + 16 * kb + 4 * l4);
    float vr[kC / 16][4][2];
#pragma unroll
    for (int kb = 0; kb < kC / 16; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* vrow =
                vv + base + (size_t)min(16 * kb + 4 * l4 + j, nt - 1) * kD + 32 * wave + l16;
            vr[kb][j][0] = vrow[0];
            vr[kb][j][1] = vrow[16];
        }
#pragma unroll
    for (int n = 0; n < kC * kD / 4 / 256; ++n) {
        const int i = tid + 256 * n, r = i / (kD / 4), c4 = i % (kD / 4);
        const f32x4 v = ld4(kk + base + (size_t)min(r, nt - 1) * kD + c4 * 4);
        st4(&Ks[r * KP + c4 * 4], r < nt ? v : f32x4{0.f, 0.f, 0.f, 0.f});
    }
    if (wave == 0) {  // cumulative log-decay and the factors formed from it
        const size_t g = tile * kC;
        const int r = min(lane, nt - 1);
        const float al = alpha[g + r], be = beta[g + r];
        float a = lane < nt ? al : 0.0f;
#pragma unroll
        for (int d = 1; d < kC; d *= 2) {
            const float o = __shfl_up(a, d);
            a = lane >= d ? a + o : a;
        }
        const float end = __shfl(a, kC - 1);
        const float b = lane < nt ? be : 0.0f;
        gs[lane] = a;
        bs[lane] = b;
        bg[lane] = b * expf(a);
        dec[lane] = lane < nt ? expf(end - a) : 0.0f;  // gamma_end / gamma_t
        Gc[g + lane] = a;
    }
    __syncthreads();

    // A = beta_t (gamma_t/gamma_s) K K^T, strictly lower: row block 3 - wave
    {
        const int tb = 3 - wave, t = 16 * tb + l16;
        f32x4 kt[kD / 16];
#pragma unroll
        for (int kb = 0; kb < kD / 16; ++kb) kt[kb] = ld4(&Ks[t * KP + 16 * kb + 4 * l4]);
        const float gt = gs[t], bt = bs[t];
        for (int sb = 0; sb <= tb; ++sb) {
            f32x4 acc[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < kD / 16; ++kb) {
                const f32x4 a = ld4(&Ks[(16 * sb + l16) * KP + 16 * kb + 4 * l4]);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = mma(a[j], kt[kb][j], acc[j]);
            }
            const f32x4 g4 = ld4(&gs[16 * sb + 4 * l4]);
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = (acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i]);
                v[i] = 16 * sb + 4 * l4 + i < t ? bt * expf(gt - g4[i]) * p : 0.0f;
            }
            st4(&Ts[t * TP + 16 * sb + 4 * l4], v);
        }
    }

    // Mq[t][s] = (gamma_t/gamma_s) q_t . k_s for s <= t: row block wave
    {
        const float gt = gs[tq];
        float* mq = Mq + tile * kC * kC + (size_t)wave * 4 * kBlk + lane * 4;
        for (int sb = 0; sb <= wave; ++sb) {
            f32x4 acc[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < kD / 16; ++kb) {
                const f32x4 a = ld4(&Ks[(16 * sb + l16) * KP + 16 * kb + 4 * l4]);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = mma(a[j], qv[kb][j], acc[j]);
            }
            const f32x4 g4 = ld4(&gs[16 * sb + 4 * l4]);
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = (acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i]);
                v[i] = (16 * sb + 4 * l4 + i <= tq && tq < nt) ? expf(gt - g4[i]) * p : 0.0f;
            }
            st4(mq + sb * kBlk, v);
        }
    }
    __syncthreads();

    // inverse of the wave's diagonal block: lane l16 column l16 (the four
    // lane groups alike), row r's value known once the rows before it have
    // been subtracted
    {
        const float* A = Ts + (16 * wave) * TP + 16 * wave;
        float* X = Xs + (16 * wave) * TP + 16 * wave + l16;
        f32x4 ar[16][4];
#pragma unroll
        for (int t = 1; t < 16; ++t)
#pragma unroll
            for (int k = 0; k < (t + 3) / 4; ++k) ar[t][k] = ld4(A + t * TP + 4 * k);
        float x[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) x[t] = t == l16 ? 1.0f : 0.0f;
#pragma unroll
        for (int r = 0; r < 15; ++r)
#pragma unroll
            for (int t = r + 1; t < 16; ++t) x[t] = fmaf(-ar[t][r / 4][r % 4], x[r], x[t]);
#pragma unroll
        for (int t = 0; t < 16; ++t)
            if (l4 == t / 4) X[t * TP] = x[t];
    }
    __syncthreads();

    // block (m, k) of A or X as an A operand, and of X as a B operand
    auto rows = [&](const float* M, int m, int k) {
        return ld4(M + (16 * m + l16) * TP + 16 * k + 4 * l4);
    };
    auto cols = [&](int k, int n) {
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = Xs[(16 * k + 4 * l4 + j) * TP + 16 * n + l16];
        return v;
    };
    auto put = [&](int m, int n, f32x4 v) {
#pragma unroll
        for (int i = 0; i < 4; ++i) Xs[(16 * m + 4 * l4 + i) * TP + 16 * n + l16] = -v[i];
    };
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    if (wave < 2) {  // 16 -> 32 rows
        const int b = 2 * wave;
        const f32x4 p = mma4(rows(Ts, b + 1, b), cols(b, b), zero);
        put(b + 1, b, mma4(rows(Xs, b + 1, b + 1), p, zero));
    }
    __syncthreads();
    {  // 32 -> 64 rows: block (m, n) of the lower left half
        const int n = wave & 1, m = 2 + (wave >> 1);
        f32x4 p2 = zero, p3 = zero;
        for (int k = n; k < 2; ++k) {
            const f32x4 x = cols(k, n);
            p2 = mma4(rows(Ts, 2, k), x, p2);
            p3 = mma4(rows(Ts, 3, k), x, p3);
        }
        f32x4 v = mma4(rows(Xs, m, 2), p2, zero);
        if (m == 3) v = mma4(rows(Xs, 3, 3), p3, v);
        put(m, n, v);
    }
    __syncthreads();

    // U = X diag(beta) V, Wk = X diag(beta gamma) K (stored negated), and
    // K^T diag(gamma_end / gamma): columns 32 wave .. + 31
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
        const int cb = 2 * wave + ct;
        f32x4 wk[4], u[4];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) wk[rt] = u[rt] = zero;
#pragma unroll
        for (int kb = 0; kb < kC / 16; ++kb) {
            const int s = 16 * kb + 4 * l4;
            const f32x4 b4 = ld4(&bs[s]), g4 = ld4(&bg[s]), d4 = ld4(&dec[s]);
            f32x4 kd, kg, vb;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float kv = Ks[(s + j) * KP + 16 * cb + l16];
                kd[j] = kv * d4[j];
                kg[j] = kv * g4[j];
                vb[j] = s + j < nt ? vr[kb][j][ct] * b4[j] : 0.0f;
            }
            st4(kk + base + (size_t)(cb * 4 + kb) * kBlk + lane * 4, kd);
#pragma unroll
            for (int rt = kb; rt < 4; ++rt) {
                const f32x4 x = rows(Xs, rt, kb);
                wk[rt] = mma4(kg, x, wk[rt]);  // transposed: rows d_k, columns t
                u[rt] = mma4(x, vb, u[rt]);
            }
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
            const size_t o = base + (size_t)(rt * 8 + cb) * kBlk + lane * 4;
            st4(Wk + o, -wk[rt]);
            st4(U + o, u[rt]);
        }
    }
}

// Per (head, 16 value columns), chunks in order:
//   W = U - Wk S,  S = gamma_end S + K^T diag(gamma_end / gamma) W.
// Only these two products depend on the state; the state before each chunk
// and W (over U) are written out for the outputs. A serial chain, bound by
// the matrix cores' time of its 64 products a SIMD and chunk and by the two
// exchanges through LDS: wave w takes row block w % 4 of W over half of K
// (w / 4; the halves meet as W is read), then row block w of the state. All
// operands arrive in operand order, kRing chunks ahead.
constexpr int kRing = 3;

__global__ __launch_bounds__(512) void k_dn_chunk_chain(
    const float* __restrict__ Kt, const float* __restrict__ Wk, float* UW,
    const float* __restrict__ Gc, int T, int H, float* __restrict__ state,
    float* __restrict__ Sall) {
    __shared__ __attribute__((aligned(16))) float Ss[8 * kBlk];
    __shared__ __attribute__((aligned(16))) float Wp[2][4 * kBlk];
    const int h = blockIdx.x, jt = blockIdx.y, jb = jt * CB;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    const int rt = wave & 3, kh = wave >> 2;
    const int nch = (T + kC - 1) / kC;
    const size_t CS = (size_t)H * kC * kD;  // a chunk of every head
    const size_t at = (size_t)h * kC * kD + lane * 4;
    const float* wk_p = Wk + at + (rt * 8 + 4 * kh) * kBlk;
    const float* kt_p = Kt + at + wave * 4 * kBlk;
    float* uw_p = UW + at + (rt * 8 + jt) * kBlk;
    float* s_p = Sall + 2 * (size_t)h * kC * kD + (jt * 8 + wave) * kBlk + lane * 4;
    const float* g_p = Gc + (size_t)h * kC + kC - 1;

    f32x4 wk[kRing][4], kt[kRing][4], u[kRing];
    float ge[kRing];
    auto load_w = [&](int s, int c) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) wk[s][kb] = ld4(wk_p + (size_t)c * CS + kb * kBlk);
        if (kh == 0) u[s] = ld4(uw_p + (size_t)c * CS);
    };
    auto load_k = [&](int s, int c) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) kt[s][kb] = ld4(kt_p + (size_t)c * CS + kb * kBlk);
        ge[s] = g_p[(size_t)c * H * kC];
    };
    float* Sg = state + (size_t)h * kD * kD + (size_t)(16 * wave + 4 * l4) * kD + jb + l16;
    f32x4 sacc;  // state rows 16 wave + 4 l4 + i, column jb + l16
#pragma unroll
    for (int i = 0; i < 4; ++i) sacc[i] = Sg[i * kD];
#pragma unroll
    for (int s = 0; s < kRing; ++s) {
        u[s] = f32x4{0.f, 0.f, 0.f, 0.f};
        load_w(s, min(s, nch - 1));
        load_k(s, min(s, nch - 1));
    }
    st4(&Ss[wave * kBlk + lane * 4], sacc);
    __syncthreads();
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < nch; c0 += kRing) {
#pragma unroll
        for (int s = 0; s < kRing; ++s) {
            const int c = c0 + s;
            if (c >= nch) break;
            const int cn = min(c + kRing, nch - 1);
            f32x4 w0 = u[s], w1 = zero;
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const f32x4 b = ld4(&Ss[(4 * kh + kb) * kBlk + lane * 4]);
                w0 = mma(wk[s][kb][0], b[0], w0);
                w1 = mma(wk[s][kb][1], b[1], w1);
                w0 = mma(wk[s][kb][2], b[2], w0);
                w1 = mma(wk[s][kb][3], b[3], w1);
            }
            st4(&Wp[kh][rt * kBlk + lane * 4], w0 + w1);
            st4(s_p + (size_t)c * 2 * CS, sacc);
            load_w(s, cn);
            __syncthreads();  // W of chunk c is in LDS, its state was read
            f32x4 d0 = sacc * expf(ge[s]), d1 = zero;
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const f32x4 b = ld4(&Wp[0][kb * kBlk + lane * 4]) + ld4(&Wp[1][kb * kBlk + lane * 4]);
                if (wave == kb) st4(uw_p + (size_t)c * CS, b);
                d0 = mma(kt[s][kb][0], b[0], d0);
                d1 = mma(kt[s][kb][1], b[1], d1);
                d0 = mma(kt[s][kb][2], b[2], d0);
                d1 = mma(kt[s][kb][3], b[3], d1);
            }
            load_k(s, cn);
            sacc = d0 + d1;
            st4(&Ss[wave * kBlk + lane * 4], sacc);
            __syncthreads();  // the state of chunk c + 1 is in LDS, W was read
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) Sg[i * kD] = sacc[i];
}

// Per (chunk, head), transposed (rows value columns, columns t):
//   O = (gamma_t (Q S) + Mq W) / sqrt(d),
// wave w value columns 32 w .. + 31 of all 64 rows; then the head RMSNorm
// (the waves' sums of squares meet in LDS) and the SiLU(z) gate, and the conv
// ring rows of the last three positions. A workgroup takes NB row blocks: all
// four, or one where the chunks are too few to fill the chip (66 rows, 16
// heads: 15.2 -> 7.2 us). V4: proj and out rows take 16-byte accesses.
template <int NB, bool V4>
__global__ __launch_bounds__(256, 2) void k_dn_chunk_out(
    const float* __restrict__ qn, const float* __restrict__ Sall, const float* __restrict__ Mq,
    const float* __restrict__ W, const float* __restrict__ Gc, const float* __restrict__ proj,
    int ldp, int T, const float* __restrict__ norm_w, float* __restrict__ out, int ldo, int H,
    float* __restrict__ conv_state, int p0) {
    __shared__ float red[4][16 * NB];
    const int c = blockIdx.x / (4 / NB), h = blockIdx.y;
    const int rb = blockIdx.x % (4 / NB) * NB;  // first row block
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    const int t0 = c * kC, nt = min(kC, T - t0);
    if (16 * rb >= nt) return;
    const int HD = H * kD, C = 3 * HD;
    const size_t tile = (size_t)c * H + h;
    const size_t base = tile * kC * kD;
    const int col = h * kD + 32 * wave + 4 * l4;  // + 16 d + i
    auto load = [&](const float* p) {
        if constexpr (V4) return ld4(p);
        else return f32x4{p[0], p[1], p[2], p[3]};
    };
    f32x4 z[2][NB];
#pragma unroll
    for (int tb = 0; tb < NB; ++tb) {
        const float* zr = proj + (size_t)(t0 + min(16 * (rb + tb) + l16, nt - 1)) * ldp + 3 * HD + col;
#pragma unroll
        for (int d = 0; d < 2; ++d) z[d][tb] = load(zr + 16 * d);
    }
    f32x4 nw[2];
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) nw[d][i] = norm_w[32 * wave + 16 * d + 4 * l4 + i];
    float g[NB];
#pragma unroll
    for (int tb = 0; tb < NB; ++tb) g[tb] = Gc[tile * kC + 16 * (rb + tb) + l16];

    f32x4 o[2][NB];
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int tb = 0; tb < NB; ++tb) o[d][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // rows past the chunk's last feed only their own columns, never stored
    const float* s_p = Sall + 2 * base + (size_t)wave * 16 * kBlk + lane * 4;
    const float* q_p = qn + base + (size_t)(16 * rb + l16) * kD + 4 * l4;
    // one row block: every operand is requested before the first product
    constexpr int PF = NB == 1 ? kD / 16 : 1;
    f32x4 sv[PF][2], qv[PF][NB];
    auto load_sq = [&](int kb) {
#pragma unroll
        for (int d = 0; d < 2; ++d) sv[kb % PF][d] = ld4(s_p + (d * 8 + kb) * kBlk);
#pragma unroll
        for (int tb = 0; tb < NB; ++tb) qv[kb % PF][tb] = ld4(q_p + 16 * tb * kD + 16 * kb);
    };
    if constexpr (PF > 1) {
#pragma unroll
        for (int kb = 0; kb < PF; ++kb) load_sq(kb);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int kb = 0; kb < kD / 16; ++kb) {
        if constexpr (PF == 1) load_sq(kb);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int tb = 0; tb < NB; ++tb)
                    o[d][tb] = mma(sv[kb % PF][d][j], qv[kb % PF][tb][j], o[d][tb]);
    }
#pragma unroll
    for (int tb = 0; tb < NB; ++tb) {
        const float gt = expf(g[tb]);
#pragma unroll
        for (int d = 0; d < 2; ++d) o[d][tb] *= gt;
    }
    const float* w_p = W + base + (size_t)2 * wave * kBlk + lane * 4;
    const float* m_p = Mq + tile * kC * kC + lane * 4;
#pragma unroll
    for (int kb = 0; kb < kC / 16; ++kb) {
        if (NB < 4 && kb >= rb + NB) break;
        f32x4 wv[2], mv[NB];
#pragma unroll
        for (int d = 0; d < 2; ++d) wv[d] = ld4(w_p + (kb * 8 + d) * kBlk);
#pragma unroll
        for (int tb = NB < 4 ? 0 : kb; tb < NB; ++tb) mv[tb] = ld4(m_p + ((rb + tb) * 4 + kb) * kBlk);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int tb = NB < 4 ? 0 : kb; tb < NB; ++tb) o[d][tb] = mma(wv[d][j], mv[tb][j], o[d][tb]);
    }
    const float rsd = 1.0f / sqrtf((float)kD);
#pragma unroll
    for (int tb = 0; tb < NB; ++tb) {
        float ss = 0.0f;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            o[d][tb] *= rsd;
#pragma unroll
            for (int i = 0; i < 4; ++i) ss = fmaf(o[d][tb][i], o[d][tb][i], ss);
        }
        ss = xor32_add(xor16_add(ss));
        if (l4 == 0) red[wave][16 * tb + l16] = ss;
    }
    __syncthreads();
#pragma unroll
    for (int tb = 0; tb < NB; ++tb) {
        const int tr = 16 * tb + l16, t = 16 * rb + tr;
        const float tot = (red[0][tr] + red[1][tr]) + (red[2][tr] + red[3][tr]);
        const float sn = 1.0f / sqrtf(tot / (float)kD + 1e-6f);
        if (t < nt) {
            float* dst = out + (size_t)(t0 + t) * ldo + col;
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                f32x4 v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = ((o[d][tb][i] * sn) * nw[d][i]) * silu_f(z[d][tb][i]);
                if constexpr (V4) {
                    st4(dst + 16 * d, v);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) dst[16 * d + i] = v[i];
                }
            }
        }
    }
    // ring row of position p0 + t: its conv input
    for (int t = max(t0 + 16 * rb, T - 3); t < t0 + min(16 * (rb + NB), nt); ++t) {
        const int row = (p0 + t) % 3;
        for (int i = tid; i < 3 * kD; i += 256) {
            const int ch = (i / kD) * HD + h * kD + i % kD;
            conv_state[(size_t)row * C + ch] = proj[(size_t)t * ldp + ch];
        }
    }
}

size_t a256(size_t b) { return (b + 255) & ~(size_t)255; }

// kn becomes the decayed K^T, U the chunks' W; the states before each chunk
// (two rows' worth) take v's place, which only the intra kernel reads, and
// the rows after it.
struct ChunkWork {
    float *qn, *kn, *U, *Wk, *vv, *alpha, *beta, *Gc, *Mq;
    size_t bytes;
};

ChunkWork carve(void* base, int T, int H) {
    ChunkWork w{};
    const int nch = (T + kC - 1) / kC;  // whole chunks
    const size_t rows = a256((size_t)nch * kC * H * kD * sizeof(float));
    const size_t sc = a256((size_t)nch * kC * H * sizeof(float));
    const size_t mq = a256((size_t)nch * H * kC * kC * sizeof(float));
    char* p = reinterpret_cast<char*>(base);
    auto take = [&](size_t b) {
        float* r = reinterpret_cast<float*>(p);
        if (p) p += b;
        return r;
    };
    w.qn = take(rows);
    w.kn = take(rows);
    w.U = take(rows);
    w.Wk = take(rows);
    w.vv = take(2 * rows);
    w.alpha = take(sc);
    w.beta = take(sc);
    w.Gc = take(sc);
    w.Mq = take(mq);
    w.bytes = 6 * rows + 3 * sc + mq;
    return w;
}

}  // namespace

extern "C" size_t qlm_deltanet_chunk_workspace_bytes(int T, int H, int d) {
    if (T <= 0 || H <= 0 || d != kD) return 0;
    return carve(nullptr, T, H).bytes;
}

extern "C" int qlm_deltanet_prefill_chunked(const float* proj, int ldp, int T, float* conv_state,
                                            const float* conv_w_t, const float* A_log,
                                            const float* dt_bias, const float* norm_w,
                                            float* state, int p0, float* out, int ldo, int H,
                                            int d, void* work, size_t work_bytes,
                                            void* stream) {
    if (!proj || !conv_state || !conv_w_t || !A_log || !dt_bias || !norm_w || !state || !out ||
        !work || T <= 0 || H <= 0 || p0 < 0)
        return QLM_ERR_ARG;
    if (d != kD) return QLM_ERR_SHAPE;
    if (ldp < 4 * H * d + 2 * H || ldo < H * d) return QLM_ERR_SHAPE;
    const ChunkWork w = carve(work, T, H);
    if (work_bytes < w.bytes || ((uintptr_t)work & 255u)) return QLM_ERR_ARG;
    hipStream_t st = as_stream(stream);
    const int nch = (T + kC - 1) / kC;
    const bool few = (long long)T * H < 8192;
    hipLaunchKernelGGL(few ? k_dn_chunk_prep<8> : k_dn_chunk_prep<16>,
                       dim3(few ? (T + 7) / 8 : (T + 15) / 16, H), dim3(3 * kD), 0, st, proj, ldp, T, conv_state,
                       conv_w_t, A_log, dt_bias, p0, H, w.qn, w.kn, w.vv, w.alpha, w.beta);
    int rc = qlm_launch_status();
    if (rc != QLM_OK) return rc;
    hipLaunchKernelGGL(k_dn_chunk_intra, dim3(nch, H), dim3(256), 0, st, w.qn, w.kn, w.vv,
                       w.alpha, w.beta, T, H, w.U, w.Wk, w.Mq, w.Gc);
    rc = qlm_launch_status();
    if (rc != QLM_OK) return rc;
    hipLaunchKernelGGL(k_dn_chunk_chain, dim3(H, kD / CB), dim3(512), 0, st, w.kn, w.Wk, w.U, w.Gc,
                       T, H, state, w.vv);
    rc = qlm_launch_status();
    if (rc != QLM_OK) return rc;
    const bool v4 = ldp % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)proj & 15u) == 0 &&
                    ((uintptr_t)out & 15u) == 0;
    // up to two workgroups a CU a chunk's row blocks go to four workgroups, which
    // read its state four times (16 heads: 300 rows 12.5 us split; 600 rows, 640
    // workgroups split, 16.2 us whole and 16.6 split)
    const bool split = nch * H * 4 <= 512;
    const auto kern = split ? (v4 ? k_dn_chunk_out<1, true> : k_dn_chunk_out<1, false>)
                            : (v4 ? k_dn_chunk_out<4, true> : k_dn_chunk_out<4, false>);
    hipLaunchKernelGGL(kern, dim3(nch * (split ? 4 : 1), H), dim3(256), 0, st, w.qn, w.vv, w.Mq, w.U,
                       w.Gc, proj, ldp, T, norm_w, out, ldo, H, conv_state, p0);
    return qlm_launch_status();
}

// Loads this file's code object on the current device now; the runtime
// otherwise loads it at the first launch of one of its kernels (4-20 ms,
// measured inside a first prefill or decode step).
hipError_t qlm_load_deltanet_chunk() {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(k_dn_chunk_chain));
}
