// Backward of the chunked gated delta-rule PRIME prefill
// (ChunkedGatedDeltaPrimeAttention, chunked_delta_prime.py:177-283), gfx950.
//
// Per (sequence, head), chunk c of C = 64 tokens with features psi_i, phi_i
// (chunked_delta_prime.py:73-87: psi = [q, q^2/sqrt2], phi = [k/|k|,
// (k^2/|k^2|)/sqrt2]), values v_i, write rates beta_i, cumulative log-decays
// g_i = sum_{m<=i} log clamp(alpha_m, 1e-5, 1), entering state S (D x 2D):
//   d_i = e^{g_i},  b_j = e^{g_63 - g_j},  a = e^{g_63},  L_ij = e^{g_i - g_j} (i >= j)
//   T   = I + [i>j] beta_j L_ij (phi_i . phi_j)            (unit lower triangular)
//   U   = V - diag(d) Phi S^T,   E = T^-1 U,   W = diag(beta) E
//   y   = M W + diag(d) Psi S^T,  M_ij = [i>=j] L_ij (psi_i . phi_j)
//   S'  = a S + W^T diag(b) Phi,  S'' = S' min(1, B / (|S'|_F + 1e-6)).
// The backward walks the chunks in reverse with the adjoint dS of the state
// leaving the chunk:
//   clamp:  dS' = s dS'' - [s < 1 or = 1] (B / (n+1e-6)^2) <dS'', S'> / n  S'
//   state:  dS_in = a dS' + (diag(d) dY)^T Psi - (diag(d) dU)^T Phi
//           dW = diag(b) Phi dS'^T + M^T dY,  dE = diag(beta) dW,
//           dU = T^-T dE,  dT = -dU E^T (strictly lower),  dV = dU
//   features: dPsi = (dM o L) Phi + diag(d) dY S,   dM = dY W^T (masked)
//           dPhi = diag(b) W dS' + (dM o L)^T Psi + (dG + dG^T) Phi - diag(d) dU S,
//           dG_ij = dT_ij beta_j L_ij
//   beta:   dbeta = rowdot(E, dW) + colsum(dT o L o G)
//   decays: dg from a, b, d, L in T and M; dlog alpha = reverse cumulative sum
//           of dg over the chunk; dalpha = dlog alpha / alpha inside the clamp
// and q, k through the feature maps (F.normalize's backward for the k
// features, eps = feat_eps).
//
// Only S and dS run along the sequence, and both recurrences are linear in the
// state but for the clamp's scalars.  With X = T^-1 [V | diag(d) Phi] = [U0 | W0],
// A_ij = M_ij beta_j and om_j = beta_j b_j:
//   S'    = a S - S Mx + R0,           Mx = W0^T diag(om) Phi, R0 = U0^T diag(om) Phi
//   dS_in = a dS' - dS' Mx^T + Q0,     Q0 = dY^T Z, Z = diag(d) Psi - A W0
// so the work is four kernels, all fp32 on MFMA (v_mfma_f32_16x16x4_f32):
//   delta_bwd_prep   per (sequence, chunk): Mx, R0, Q0 and T^-1 as the chunk's record
//   delta_bwd_chain  per sequence, chunks in order: the states entering every chunk
//   delta_bwd_chain  per sequence, chunks in reverse: dS' of every chunk
//   delta_bwd_grad   per (sequence, chunk): every gradient from S, dS' and T^-1
// Only the chains are serial (one 128 x 128 product a chunk); the rest fills the
// chip with (sequence, chunk) workgroups.  Measured at 24 sequences of 1024
// tokens: prep 79 us, chains 97 and 115 us (6 and 7 us a chunk; the product's 128
// MFMAs a wave are 3.4 us), grad 82 us: 0.37 ms.  As one kernel per sequence, fp32
// on the VALU with the chunks in reverse and 24 of 256 CUs busy, it took 6.43 ms.

#include <algorithm>

#include "f32_common.h"

namespace prime {
namespace {

constexpr int kP = 2 * kD;       // features
constexpr int kW = 8;            // waves per workgroup of every kernel here
constexpr int kPF = kP + 4;      // 128-wide rows: 16-byte reads of 16 rows fall on distinct bank quads
constexpr int kPN = kC + 4;      // 64-wide rows
constexpr int kPX = 3 * kD + 16; // X rows: scalar reads of 4 rows x 16 columns meet no bank twice
constexpr int kPS = 32 + 4;      // the chain's state rows in operand order
constexpr float kInvSqrt2 = 0.70710678118654752f;

// four floats of a caller's state or gradient, which is only known to be 4-byte aligned
// (one 16-byte access all the same: global memory takes any dword boundary)
typedef f32x4 f32x4_dw __attribute__((aligned(4)));
__device__ __forceinline__ f32x4 ld4_dw(const float *p) { return *reinterpret_cast<const f32x4_dw *>(p); }
__device__ __forceinline__ void st4_dw(float *p, f32x4 v) { *reinterpret_cast<f32x4_dw *>(p) = v; }

// Record of one (sequence, chunk), bytes.  The chains' 128 x 128 operands are
// stored in the order they are read: [8 row blocks][64 lanes][32 k-steps], lane
// l of block b holding row 16 b + l%16, columns 32 (l/16) + s; R0 and Q0 as
// transposed accumulator tiles [8 feature blocks][4 value blocks][64 lanes][4].
constexpr int kRMT = 0;          // -Mx^T (forward chain)
constexpr int kRM = 65536;       // -Mx (reverse chain)
constexpr int kRR0 = 131072;
constexpr int kRQ0 = 163840;
constexpr int kRTI = 196608;     // T^-1, row-major 64 x 64
constexpr int kRSC = 212992;     // e^cum_63
constexpr size_t kRecB = 213248;
constexpr size_t kStB = static_cast<size_t>(kD) * kP * 4;

// Workspace of one sequence: records, the NC + 1 states (those entering each
// chunk, then the final one), dS' of each chunk, and per chunk the clamp's scale
// and the norm it was formed from.
struct SeqWs {
    uint8_t *rec;
    float *st, *ds, *sc;
};
__host__ __device__ inline size_t seq_ws_bytes(int NC) {
    return (NC * (kRecB + 2 * kStB) + kStB + static_cast<size_t>(NC) * 8 + 255) & ~static_cast<size_t>(255);
}
__device__ __forceinline__ SeqWs seq_ws(const DeltaBwdArgs &a, int slot, int NC) {
    uint8_t *p = reinterpret_cast<uint8_t *>(a.ws) + static_cast<size_t>(slot) * seq_ws_bytes(NC);
    SeqWs w;
    w.rec = p;
    w.st = reinterpret_cast<float *>(p + NC * kRecB);
    w.ds = w.st + static_cast<size_t>(NC + 1) * kD * kP;
    w.sc = w.ds + static_cast<size_t>(NC) * kD * kP;
    return w;
}

// 8 consecutive inputs of one row as fp32, zero when !valid
template <int DT>
__device__ __forceinline__ void load_row8(const void *p, int64_t off, bool valid, f32x4 &x, f32x4 &y) {
    x = y = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!valid) return;
    if constexpr (DT == PRIME_BF16) {
        const u32x4 s = *reinterpret_cast<const u32x4 *>(static_cast<const uint16_t *>(p) + off);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            x[2 * i] = __uint_as_float(s[i] << 16);
            x[2 * i + 1] = __uint_as_float(s[i] & 0xFFFF0000u);
            y[2 * i] = __uint_as_float(s[2 + i] << 16);
            y[2 * i + 1] = __uint_as_float(s[2 + i] & 0xFFFF0000u);
        }
    } else {
        x = ld4(static_cast<const float *>(p) + off);
        y = ld4(static_cast<const float *>(p) + off + 4);
    }
}
template <int DT>
__device__ __forceinline__ float load1(const void *p, int64_t off) {
    if constexpr (DT == PRIME_BF16) return bf16_bits_to_f32(static_cast<const uint16_t *>(p)[off]);
    else return static_cast<const float *>(p)[off];
}

// The chunk's features and dy in LDS (8 threads a token, 8 dims each; rows past
// L zero), the reciprocal norms of k and k^2 (sR1, sR2, where given) and, by
// wave 0, the decays and rates: cum, d = e^cum, b = e^(cum_63 - cum), beta.
template <int DT>
__device__ __forceinline__ void load_chunk(const DeltaBwdArgs &a, int seq, int c, int tid, float (*sPhi)[kPF],
                                           float (*sPsi)[kPF], float *sCum, float *sEc, float *sB, float *sBeta,
                                           float *sR1, float *sR2) {
    const int b = seq / a.H, h = seq - b * a.H, hk = h / a.group;
    const int i = tid >> 3, d0 = 8 * (tid & 7);
    const int t = c * kC + i;
    const bool valid = t < a.L;
    const int64_t tc = valid ? t : 0;
    f32x4 q[2], k[2];
    load_row8<DT>(a.q, b * a.q_sb + h * a.q_sh + tc * a.q_sl + d0, valid, q[0], q[1]);
    load_row8<DT>(a.k, b * a.k_sb + hk * a.k_sh + tc * a.k_sl + d0, valid, k[0], k[1]);
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float k2 = k[j][r] * k[j][r];
            s1 += k2;
            s2 += k2 * k2;
        }
    s1 += xor_lane<1>(s1);
    s1 += xor_lane<2>(s1);
    s1 += xor_lane<4>(s1);
    s2 += xor_lane<1>(s2);
    s2 += xor_lane<2>(s2);
    s2 += xor_lane<4>(s2);
    const float r1 = 1.0f / fmaxf(sqrtf(s1), a.feat_eps), r2 = 1.0f / fmaxf(sqrtf(s2), a.feat_eps);
    if (sR1 && (tid & 7) == 0) {
        sR1[i] = r1;
        sR2[i] = r2;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        f32x4 p1, p2, q2;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p1[r] = k[j][r] * r1;
            p2[r] = k[j][r] * k[j][r] * (r2 * kInvSqrt2);
            q2[r] = q[j][r] * q[j][r] * kInvSqrt2;
        }
        st4(&sPhi[i][d0 + 4 * j], p1);
        st4(&sPhi[i][kD + d0 + 4 * j], p2);
        st4(&sPsi[i][d0 + 4 * j], q[j]);
        st4(&sPsi[i][kD + d0 + 4 * j], q2);
    }
    if (tid < kWave) {
        const bool vl = c * kC + tid < a.L;
        const size_t o = static_cast<size_t>(seq) * a.L + c * kC + tid;
        const float bt = vl ? a.beta[o] : 0.f;
        const float al = vl ? a.alpha[o] : a.decay_pad;
        const float cum = wave_prefix_sum(logf(fminf(fmaxf(al, 1e-5f), 1.0f)));
        const float cend = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cum), 63));
        sCum[tid] = cum;
        sEc[tid] = expf(cum);
        sB[tid] = expf(cend - cum);
        sBeta[tid] = bt;
    }
}

__device__ __forceinline__ void load_dy(const DeltaBwdArgs &a, int seq, int c, int tid, f32x4 &x, f32x4 &y) {
    const int b = seq / a.H, h = seq - b * a.H;
    const int t = c * kC + (tid >> 3);
    const bool valid = t < a.L;
    const int64_t off = b * a.dy_sb + h * a.dy_sh + (valid ? t : 0) * a.dy_sl + 8 * (tid & 7);
    if (a.dt_dy == PRIME_BF16) load_row8<PRIME_BF16>(a.dy, off, valid, x, y);
    else load_row8<PRIME_F32>(a.dy, off, valid, x, y);
}

// sums over the 16 lanes of a column group (the tile's columns), in every lane
__device__ __forceinline__ float sum_cols(float x) {
    x += xor_lane<1>(x);
    x += xor_lane<2>(x);
    x += xor_lane<4>(x);
    return x + xor_lane<8>(x);
}
// sums over the four lane groups (the tile's rows beyond a lane's four)
__device__ __forceinline__ float sum_rows(float x) { return sum_lane32(sum_lane16(x)); }

}  // namespace

// ---------------------------------------------------------------------------
// Per (sequence, chunk): the chains' operands and T^-1.  The 256 columns of
// T^-1 [V | diag(d) Phi | I] are solved one per thread (the identity's columns
// take the fourth wave, idle in a 192-column solve).
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(kW *kWave, 1) void delta_bwd_prep_kernel(const DeltaBwdArgs a) {
    __shared__ __attribute__((aligned(16))) float sPhi[kC][kPF];
    __shared__ __attribute__((aligned(16))) float sPsi[kC][kPF];
    __shared__ __attribute__((aligned(16))) float sN[kC][kPN];  // N (strictly lower), then dY
    __shared__ __attribute__((aligned(16))) float sA[kC][kPN];  // A (lower tiles), then A^T dY
    __shared__ __attribute__((aligned(16))) float sX[kC][kPX];  // [U0 | W0], one row per token
    __shared__ float sCum[kC], sEc[kC], sB[kC], sBeta[kC];

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, c16 = lane & 15;
    const int NC = (a.L + kC - 1) / kC;
    const int slot = blockIdx.x / NC, c = blockIdx.x - slot * NC;
    const int seq = a.seq0 + slot;
    const int b = seq / a.H, h = seq - b * a.H, hk = h / a.group;
    uint8_t *rec = seq_ws(a, slot, NC).rec + c * kRecB;

    load_chunk<DT>(a, seq, c, tid, sPhi, sPsi, sCum, sEc, sB, sBeta, nullptr, nullptr);
    f32x4 dy0, dy1;
    load_dy(a, seq, c, tid, dy0, dy1);
    __syncthreads();

    // ---- N and A on the 10 lower tiles (feature k-slot g of k-step s: 32 g + s)
    for (int ti = w; ti < 10; ti += kW) {
        int ib, jb;
        lower_tile(ti, ib, jb);
        const float *pa = &sPhi[16 * ib + c16][32 * g];
        const float *sa = &sPsi[16 * ib + c16][32 * g];
        const float *pb = &sPhi[16 * jb + c16][32 * g];
        f32x4 gr = {0.f, 0.f, 0.f, 0.f}, ga = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q4 = 0; q4 < 8; ++q4) {
            const f32x4 x = ld4(pa + 4 * q4), y = ld4(sa + 4 * q4), z = ld4(pb + 4 * q4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                gr = mfma4(x[r], z[r], gr);
                ga = mfma4(y[r], z[r], ga);
            }
        }
        const int j = 16 * jb + c16;
        const float cj = sCum[j], bj = sBeta[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * ib + 4 * g + r;
            const float lam = i >= j ? expf(sCum[i] - cj) * bj : 0.f;
            sN[i][j] = i > j ? lam * gr[r] : 0.f;
            sA[i][j] = lam * ga[r];
        }
    }
    __syncthreads();

    if (tid < 4 * kC) {
        float x[kC];
        if (tid < kD) {
            const int64_t vo = b * a.v_sb + hk * a.v_sh + tid;
#pragma unroll
            for (int i = 0; i < kC; ++i) {
                const int t = c * kC + i;
                x[i] = t < a.L ? load1<DT>(a.v, vo + static_cast<int64_t>(t) * a.v_sl) : 0.f;
            }
        } else if (tid < kD + kP) {
#pragma unroll
            for (int i = 0; i < kC; ++i) x[i] = sEc[i] * sPhi[i][tid - kD];
        } else {
#pragma unroll
            for (int i = 0; i < kC; ++i) x[i] = i == tid - kD - kP ? 1.f : 0.f;
        }
        solve_unit_lower<kPN>(&sN[0][0], x);
        if (tid < kD + kP) {
#pragma unroll
            for (int i = 0; i < kC; ++i) sX[i][tid] = x[i];
        } else {
            float *ti = reinterpret_cast<float *>(rec + kRTI) + (tid - kD - kP);
#pragma unroll
            for (int i = 0; i < kC; ++i) ti[i * kC] = x[i];
        }
    }
    __syncthreads();
    st4(&sN[tid >> 3][8 * (tid & 7)], dy0);
    st4(&sN[tid >> 3][8 * (tid & 7) + 4], dy1);

    // wave w: feature block w as the output's rows (R0^T, -Mx^T) or columns (-Mx)
    float om[16];  // om_j of this lane's k-slots j = 4 s + g
#pragma unroll
    for (int s = 0; s < 16; ++s) om[s] = sBeta[4 * s + g] * sB[4 * s + g];
    {
        float pf[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) pf[s] = om[s] * sPhi[4 * s + g][16 * w + c16];
#pragma unroll
        for (int dv = 0; dv < 4; ++dv) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 16; ++s) acc = mfma4(pf[s], sX[4 * s + g][16 * dv + c16], acc);
            st4(rec + kRR0 + ((w * 4 + dv) * 64 + lane) * 16, acc);
        }
#pragma unroll 2
        for (int e = 0; e < 8; ++e) {
            // Mx rows f' in block e, columns f in block w, both ways round
            f32x4 m = {0.f, 0.f, 0.f, 0.f}, mt = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                const float x = sX[4 * s + g][kD + 16 * e + c16];
                m = mfma4(x, pf[s], m);    // m[r] = Mx[16 e + 4 g + r][16 w + c16]
                mt = mfma4(pf[s], x, mt);  // mt[r] = Mx[16 e + c16][16 w + 4 g + r]
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                m[r] = -m[r];
                mt[r] = -mt[r];
            }
            st4(rec + kRMT + ((w * 64 + 16 * (e >> 1) + c16) * 32 + 16 * (e & 1) + 4 * g) * 4, m);
            st4(rec + kRM + ((e * 64 + 16 * (w >> 1) + c16) * 32 + 16 * (w & 1) + 4 * g) * 4, mt);
        }
    }
    __syncthreads();  // dY staged
    // ---- A^T dY (rows j in block w/2, two value blocks; A is zero above its diagonal)
    f32x4 bt[2];
    {
        const int jb = w >> 1;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int dv = 2 * (w & 1) + jj;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            for (int s = 4 * jb; s < 16; ++s) acc = mfma4(sA[4 * s + g][16 * jb + c16], sN[4 * s + g][16 * dv + c16], acc);
            bt[jj] = acc;
        }
    }
    __syncthreads();
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int r = 0; r < 4; ++r) sA[16 * (w >> 1) + 4 * g + r][16 * (2 * (w & 1) + jj) + c16] = bt[jj][r];
    __syncthreads();
    // ---- Q0^T tiles (feature block w) = Psi^T diag(d) dY - W0^T (A^T dY)
    {
        float ps[16], wx[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            ps[s] = sEc[4 * s + g] * sPsi[4 * s + g][16 * w + c16];
            wx[s] = -sX[4 * s + g][kD + 16 * w + c16];
        }
#pragma unroll
        for (int dv = 0; dv < 4; ++dv) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 16; ++s) acc = mfma4(ps[s], sN[4 * s + g][16 * dv + c16], acc);
#pragma unroll
            for (int s = 0; s < 16; ++s) acc = mfma4(wx[s], sA[4 * s + g][16 * dv + c16], acc);
            st4(rec + kRQ0 + ((w * 4 + dv) * 64 + lane) * 16, acc);
        }
    }
    if (tid == 0) *reinterpret_cast<float *>(rec + kRSC) = sEc[kC - 1];
}

// ---------------------------------------------------------------------------
// The serial chains, one workgroup of 8 waves per sequence: wave w carries the
// state's feature block w (S^T tiles for the four value blocks in accumulators)
// and the state goes round through LDS in the operand order
// sS[dv][16 g + c][s] = S^T[32 g + s][16 dv + c].  Records are read one chunk
// ahead.  Forward: x = a S - Mx^T S + R0, its norm, the clamp's scale (applied
// in the next chunk's products: one barrier a chunk).  Reverse: dS'' to dS' by
// the clamp's derivative (an inner product with the chunk's final state, only
// where the clamp held), then x = a dS' - Mx dS' + Q0.
// ---------------------------------------------------------------------------
namespace {

struct ChainRec {
    f32x4 m[8];   // the 128 x 128 operand, k-steps 4q .. 4q+3
    f32x4 c0[4];  // R0 or Q0 tiles of feature block w
    float e63;
};

template <bool REV>
__device__ __forceinline__ void load_rec(ChainRec &R, const uint8_t *rc, int w, int lane) {
#pragma unroll
    for (int q = 0; q < 8; ++q) R.m[q] = ld4(rc + (REV ? kRM : kRMT) + ((w * 64 + lane) * 32 + 4 * q) * 4);
#pragma unroll
    for (int dv = 0; dv < 4; ++dv) R.c0[dv] = ld4(rc + (REV ? kRQ0 : kRR0) + ((w * 4 + dv) * 64 + lane) * 16);
    R.e63 = *reinterpret_cast<const float *>(rc + kRSC);
}

// x = e63 st + m (the state in sS), per value block
__device__ __forceinline__ void chain_product(const ChainRec &R, const float (*sS)[64][kPS], int lane, f32x4 (&st)[4]) {
#pragma unroll
    for (int dv = 0; dv < 4; ++dv) st[dv] *= R.e63;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        f32x4 so[4];
#pragma unroll
        for (int dv = 0; dv < 4; ++dv) so[dv] = ld4(&sS[dv][lane][4 * q]);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int dv = 0; dv < 4; ++dv) st[dv] = mfma4(R.m[q][r], so[dv][r], st[dv]);
    }
}

}  // namespace

template <bool REV>
__global__ __launch_bounds__(kW *kWave, 1) void delta_bwd_chain_kernel(const DeltaBwdArgs a) {
    __shared__ __attribute__((aligned(16))) float sS[2][4][64][kPS];
    __shared__ float sRed[2][kW];

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, c16 = lane & 15;
    const int NC = (a.L + kC - 1) / kC;
    const int slot = blockIdx.x, seq = a.seq0 + slot;
    const SeqWs ws = seq_ws(a, slot, NC);
    // this lane's elements of a [d][f] state: d = 16 dv + c16, f = 16 w + 4 g .. +3
    const int so = c16 * kP + 16 * w + 4 * g;
    const size_t sofs = static_cast<size_t>(seq) * kD * kP;
    const float *src = REV ? a.dstate_out : a.state_in;

    f32x4 st[4];
#pragma unroll
    for (int dv = 0; dv < 4; ++dv) st[dv] = src ? ld4_dw(src + sofs + so + 16 * dv * kP) : f32x4{0.f, 0.f, 0.f, 0.f};

    auto publish = [&](int buf) {
#pragma unroll
        for (int dv = 0; dv < 4; ++dv) st4(&sS[buf][dv][16 * (w >> 1) + c16][16 * (w & 1) + 4 * g], st[dv]);
    };
    auto total = [&](int buf) {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < kW; ++i) t += sRed[buf][i];
        return t;
    };

    if constexpr (!REV) {
        float sc = 1.0f;
        publish(0);
        __syncthreads();
        auto step = [&](int c, const ChainRec &R, ChainRec &nxt) {
            load_rec<REV>(nxt, ws.rec + min(c + 1, NC - 1) * kRecB, w, lane);
            float *o = ws.st + static_cast<size_t>(c) * kD * kP + so;
#pragma unroll
            for (int dv = 0; dv < 4; ++dv) st4(o + 16 * dv * kP, st[dv] * sc);
            chain_product(R, sS[c & 1], lane, st);
            float ss = 0.f;
#pragma unroll
            for (int dv = 0; dv < 4; ++dv)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    st[dv][r] = sc * st[dv][r] + R.c0[dv][r];
                    ss += st[dv][r] * st[dv][r];
                }
            publish((c & 1) ^ 1);
            ss = wave_sum(ss);
            if (lane == 0) sRed[c & 1][w] = ss;
            __syncthreads();
            const float nrm = sqrtf(total(c & 1));
            sc = a.bound > 0.f ? fminf(1.0f, a.bound / (nrm + 1e-6f)) : 1.0f;
            if (tid == 0) {
                ws.sc[2 * c] = sc;
                ws.sc[2 * c + 1] = nrm;
            }
        };
        ChainRec ra, rb;
        load_rec<REV>(ra, ws.rec, w, lane);
        int c = 0;
        for (; c + 1 < NC; c += 2) {
            step(c, ra, rb);
            step(c + 1, rb, ra);
        }
        if (c < NC) step(c, ra, rb);
        float *o = ws.st + static_cast<size_t>(NC) * kD * kP + so;
#pragma unroll
        for (int dv = 0; dv < 4; ++dv) st4(o + 16 * dv * kP, st[dv] * sc);
    } else {
        // the chunk's final state and its clamp, read one chunk ahead
        struct Fin {
            f32x4 s[4];
            float sc, nrm;
        };
        auto load_fin = [&](Fin &F, int c) {
            const float *p = ws.st + static_cast<size_t>(c + 1) * kD * kP + so;
#pragma unroll
            for (int dv = 0; dv < 4; ++dv) F.s[dv] = ld4(p + 16 * dv * kP);
            F.sc = ws.sc[2 * c];
            F.nrm = ws.sc[2 * c + 1];
        };
        auto step = [&](int c, const ChainRec &R, ChainRec &nxt, const Fin &F, Fin &fnxt) {
            const int cn = max(c - 1, 0), buf = c & 1;
            load_rec<REV>(nxt, ws.rec + cn * kRecB, w, lane);
            load_fin(fnxt, cn);
            const float x = a.bound / (F.nrm + 1e-6f);
            if (a.bound > 0.f && x <= 1.0f) {  // (the same for every lane)
                float c1 = 0.f;
#pragma unroll
                for (int dv = 0; dv < 4; ++dv)
#pragma unroll
                    for (int r = 0; r < 4; ++r) c1 = fmaf(st[dv][r], F.s[dv][r], c1);
                c1 = wave_sum(c1);
                if (lane == 0) sRed[buf][w] = c1;
                __syncthreads();
                // <dS'', S'> = <dS'', S''> / x; dS' = x dS'' - B <dS'', S'> / ((n + 1e-6)^2 n) S'
                const float den = F.nrm + 1e-6f;
                const float coef = -a.bound / (den * den) * (total(buf) / x) / F.nrm / x;
#pragma unroll
                for (int dv = 0; dv < 4; ++dv) st[dv] = x * st[dv] + coef * F.s[dv];
            }
            publish(buf);
            float *o = ws.ds + static_cast<size_t>(c) * kD * kP + so;
#pragma unroll
            for (int dv = 0; dv < 4; ++dv) st4(o + 16 * dv * kP, st[dv]);
            __syncthreads();
            chain_product(R, sS[buf], lane, st);
#pragma unroll
            for (int dv = 0; dv < 4; ++dv) st[dv] += R.c0[dv];
        };
        ChainRec ra, rb;
        Fin fa, fb;
        load_rec<REV>(ra, ws.rec + (NC - 1) * kRecB, w, lane);
        load_fin(fa, NC - 1);
        int c = NC - 1;
        for (; c >= 1; c -= 2) {
            step(c, ra, rb, fa, fb);
            step(c - 1, rb, ra, fb, fa);
        }
        if (c == 0) step(0, ra, rb, fa, fb);
        if (a.dstate_in) {
#pragma unroll
            for (int dv = 0; dv < 4; ++dv) st4_dw(a.dstate_in + sofs + so + 16 * dv * kP, st[dv]);
        }
    }
}

// ---------------------------------------------------------------------------
// Per (sequence, chunk): every gradient, from the state S entering the chunk,
// dS' and T^-1.  8 waves; wave w owns token block w/2 and half w%2 of the value
// or feature blocks of each product, and tiles w and w + 8 of the 10 lower tiles.
// The dPsi and dPhi tiles (features x tokens) stay in accumulators throughout;
// the C x C and C x D operands share LDS buffers in turn (157 KB in all), each
// change of a buffer's contents between two barriers.
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(kW *kWave, 1) void delta_bwd_grad_kernel(const DeltaBwdArgs a) {
    __shared__ __attribute__((aligned(16))) float sPhi[kC][kPF];
    __shared__ __attribute__((aligned(16))) float sPsi[kC][kPF];
    __shared__ __attribute__((aligned(16))) float sSt[kD][kPF];  // S, dS', S
    __shared__ __attribute__((aligned(16))) float sY[kC][kPN];   // dY, then dM o L (lower tiles)
    __shared__ __attribute__((aligned(16))) float sE[kC][kPN];   // E, then dG + dG^T
    __shared__ __attribute__((aligned(16))) float sT[kC][kPN];   // U, M (lower tiles), dE, dU
    __shared__ float sCum[kC], sEc[kC], sB[kC], sBeta[kC], sR1[kC], sR2[kC];
    __shared__ float sZ[2][kC], sDb[2][kC], sDp[2][kC], sDh[2][kC];  // row sums, one per half
    __shared__ float sTr[10][16], sTc[10][16], sTb[10][16];         // the lower tiles' row and column sums
    __shared__ float sRed[kW];

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, c16 = lane & 15;
    const int ib = w >> 1, hb = w & 1;
    const int tok = 16 * ib + c16;  // the token of this lane's feature tiles
    const int NC = (a.L + kC - 1) / kC;
    const int slot = blockIdx.x / NC, c = blockIdx.x - slot * NC;
    const int seq = a.seq0 + slot;
    const int b = seq / a.H, h = seq - b * a.H, hk = h / a.group;
    const SeqWs ws = seq_ws(a, slot, NC);
    const uint8_t *rec = ws.rec + c * kRecB;
    const float *ti = reinterpret_cast<const float *>(rec + kRTI);
    const int t0 = c * kC;
    const size_t obase = static_cast<size_t>(seq) * a.L + t0;

    // state rows d = tid / 8, features 16 (tid % 8) .. +15
    f32x4 sreg[4], dreg[4];
    {
        const int o = (tid >> 3) * kP + 16 * (tid & 7);
        const float *p = ws.st + static_cast<size_t>(c) * kD * kP + o, *d = ws.ds + static_cast<size_t>(c) * kD * kP + o;
#pragma unroll
        for (int i = 0; i < 4; ++i) sreg[i] = ld4(p + 4 * i);
#pragma unroll
        for (int i = 0; i < 4; ++i) dreg[i] = ld4(d + 4 * i);
    }
    auto put_state = [&](const f32x4 (&x)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) st4(&sSt[tid >> 3][16 * (tid & 7) + 4 * i], x[i]);
    };
    // T^-1 operands: rows of this token block (k = 16 g + s), and its columns (k = 4 s + g)
    f32x4 tr[4];
    float tt[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) tr[q] = ld4(ti + (16 * ib + c16) * kC + 16 * g + 4 * q);
#pragma unroll
    for (int s = 0; s < 16; ++s) tt[s] = ti[(4 * s + g) * kC + 16 * ib + c16];

    load_chunk<DT>(a, seq, c, tid, sPhi, sPsi, sCum, sEc, sB, sBeta, sR1, sR2);
    {
        f32x4 x, y;
        load_dy(a, seq, c, tid, x, y);
        st4(&sY[tid >> 3][8 * (tid & 7)], x);
        st4(&sY[tid >> 3][8 * (tid & 7) + 4], y);
    }
    put_state(sreg);
    {
        float t = 0.f;  // <dS', S>
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) t = fmaf(dreg[i][r], sreg[i][r], t);
        t = wave_sum(t);
        if (lane == 0) sRed[w] = t;
    }
    __syncthreads();

    // ---- U = V - diag(d) Phi S^T (tiles tokens x values)
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
        const int db = 2 * hb + jj;
        const float *pa = &sPhi[16 * ib + c16][32 * g], *pb = &sSt[16 * db + c16][32 * g];
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const f32x4 x = ld4(pa + 4 * q), z = ld4(pb + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc = mfma4(x[r], z[r], acc);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * ib + 4 * g + r;
            const float v = t0 + i < a.L ? load1<DT>(a.v, b * a.v_sb + hk * a.v_sh +
                                                              static_cast<int64_t>(t0 + i) * a.v_sl + 16 * db + c16)
                                         : 0.f;
            sT[i][16 * db + c16] = v - sEc[i] * acc[r];
        }
    }
    // ---- dPsi from the readout of S: d_i S^T dy_i, and its share of dg
    f32x4 dpsi[2][2], dphi[2][2];  // [feature block in the half][k or q, squares]
    const float ec = sEc[tok];
    {
        float dot = 0.f;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int fb = 2 * hb + jj + 4 * hf;
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
                for (int s = 0; s < 16; ++s) acc = mfma4(sSt[4 * s + g][16 * fb + c16], sY[tok][4 * s + g], acc);
                const f32x4 p = ld4(&sPsi[tok][16 * fb + 4 * g]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc[r] *= ec;
                    dot = fmaf(p[r], acc[r], dot);
                }
                dpsi[jj][hf] = acc;
            }
        dot = sum_rows(dot);
        if (g == 0) sDp[hb][tok] = dot;
    }
    // ---- the lower tiles: L, L o G (i > j), M = L o (psi . phi)
    f32x4 lt[2], lg[2], mm[2], dm[2], xs[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        if (w + kW * n >= 10) break;
        int tib, tjb;
        lower_tile(w + kW * n, tib, tjb);
        const float *pa = &sPhi[16 * tib + c16][32 * g], *sa = &sPsi[16 * tib + c16][32 * g];
        const float *pb = &sPhi[16 * tjb + c16][32 * g];
        f32x4 gr = {0.f, 0.f, 0.f, 0.f}, ga = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const f32x4 x = ld4(pa + 4 * q), y = ld4(sa + 4 * q), z = ld4(pb + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                gr = mfma4(x[r], z[r], gr);
                ga = mfma4(y[r], z[r], ga);
            }
        }
        const int j = 16 * tjb + c16;
        const float cj = sCum[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * tib + 4 * g + r;
            lt[n][r] = i >= j ? expf(sCum[i] - cj) : 0.f;
            lg[n][r] = i > j ? lt[n][r] * gr[r] : 0.f;
            mm[n][r] = lt[n][r] * ga[r];
        }
    }
    __syncthreads();

    // ---- E = T^-1 U; dS' takes S's place
    put_state(dreg);
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
        const int db = 2 * hb + jj;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc = mfma4(tr[q][r], sT[16 * g + 4 * q + r][16 * db + c16], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) sE[16 * ib + 4 * g + r][16 * db + c16] = acc[r];
    }
    __syncthreads();

    // ---- dM = beta_j (dY_i . E_j) on the lower tiles; M into LDS (U is consumed)
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        if (w + kW * n >= 10) break;
        int tib, tjb;
        lower_tile(w + kW * n, tib, tjb);
        f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 x = ld4(&sY[16 * tib + c16][16 * g + 4 * q]), z = ld4(&sE[16 * tjb + c16][16 * g + 4 * q]);
#pragma unroll
            for (int r = 0; r < 4; ++r) p = mfma4(x[r], z[r], p);
        }
        const int j = 16 * tjb + c16;
        const float bj = sBeta[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float d = bj * p[r];
            xs[n][r] = d * mm[n][r];  // dM_ij M_ij (M is zero above the diagonal)
            dm[n][r] = d * lt[n][r];
            sT[16 * tib + 4 * g + r][j] = mm[n][r];
        }
    }
    __syncthreads();

    // ---- dW = diag(b) Phi dS'^T + M^T dY (tiles tokens x values), its row products with E, dE
    f32x4 de[2];
    {
        float z[4] = {0.f, 0.f, 0.f, 0.f}, zb[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int db = 2 * hb + jj;
            const float *pa = &sPhi[16 * ib + c16][32 * g], *pb = &sSt[16 * db + c16][32 * g];
            f32x4 p2 = {0.f, 0.f, 0.f, 0.f}, my = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const f32x4 x = ld4(pa + 4 * q), y = ld4(pb + 4 * q);
#pragma unroll
                for (int r = 0; r < 4; ++r) p2 = mfma4(x[r], y[r], p2);
            }
            for (int s = 4 * ib; s < 16; ++s) my = mfma4(sT[4 * s + g][16 * ib + c16], sY[4 * s + g][16 * db + c16], my);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = 16 * ib + 4 * g + r;
                const float e = sE[j][16 * db + c16], dws = sB[j] * p2[r], dw = dws + my[r];
                z[r] = fmaf(e, dws, z[r]);
                zb[r] = fmaf(e, dw, zb[r]);
                de[jj][r] = sBeta[j] * dw;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float x = sum_cols(z[r]), y = sum_cols(zb[r]);
            if (c16 == 0) {
                sZ[hb][16 * ib + 4 * g + r] = x;
                sDb[hb][16 * ib + 4 * g + r] = y;
            }
        }
    }
    // ---- dPhi from dS': b_j beta_j dS'^T E_j
    {
        const float om = sB[tok] * sBeta[tok];
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int fb = 2 * hb + jj + 4 * hf;
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
                for (int s = 0; s < 16; ++s) acc = mfma4(sSt[4 * s + g][16 * fb + c16], sE[tok][4 * s + g], acc);
                dphi[jj][hf] = acc * om;
            }
    }
    __syncthreads();
    // ---- dE for M, dM o L for dY, S for dS'
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int r = 0; r < 4; ++r) sT[16 * ib + 4 * g + r][16 * (2 * hb + jj) + c16] = de[jj][r];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        if (w + kW * n >= 10) break;
        int tib, tjb;
        lower_tile(w + kW * n, tib, tjb);
#pragma unroll
        for (int r = 0; r < 4; ++r) sY[16 * tib + 4 * g + r][16 * tjb + c16] = dm[n][r];
    }
    put_state(sreg);
    __syncthreads();

    // ---- dU = T^-T dE (= dV); dPsi += (dM o L) Phi, dPhi += (dM o L)^T Psi
    f32x4 du[2];
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
        const int db = 2 * hb + jj;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 16; ++s) acc = mfma4(tt[s], sT[4 * s + g][16 * db + c16], acc);
        du[jj] = acc;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = 16 * ib + 4 * g + r;
            if (t0 + j < a.L) a.dv[(obase + j) * kD + 16 * db + c16] = acc[r];
        }
    }
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const int fb = 2 * hb + jj + 4 * hf;
            f32x4 x = dpsi[jj][hf], y = dphi[jj][hf];
            for (int s = 0; s < 4 * (ib + 1); ++s) x = mfma4(sPhi[4 * s + g][16 * fb + c16], sY[tok][4 * s + g], x);
            for (int s = 4 * ib; s < 16; ++s) y = mfma4(sPsi[4 * s + g][16 * fb + c16], sY[4 * s + g][tok], y);
            dpsi[jj][hf] = x;
            dphi[jj][hf] = y;
        }
    __syncthreads();
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int r = 0; r < 4; ++r) sT[16 * ib + 4 * g + r][16 * (2 * hb + jj) + c16] = du[jj][r];
    __syncthreads();

    // ---- dPhi -= d_i S^T du_i, and its share of dg
    {
        float dot = 0.f;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int fb = 2 * hb + jj + 4 * hf;
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
                for (int s = 0; s < 16; ++s) acc = mfma4(sSt[4 * s + g][16 * fb + c16], sT[tok][4 * s + g], acc);
                const f32x4 p = ld4(&sPhi[tok][16 * fb + 4 * g]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc[r] *= -ec;
                    dot = fmaf(p[r], acc[r], dot);
                }
                dphi[jj][hf] += acc;
            }
        dot = sum_rows(dot);
        if (g == 0) sDh[hb][tok] = dot;
    }
    // ---- dT = -dU E^T (i > j) on the lower tiles: dg, dbeta, dG
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        if (w + kW * n >= 10) break;
        int tib, tjb;
        lower_tile(w + kW * n, tib, tjb);
        f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 x = ld4(&sT[16 * tib + c16][16 * g + 4 * q]), z = ld4(&sE[16 * tjb + c16][16 * g + 4 * q]);
#pragma unroll
            for (int r = 0; r < 4; ++r) p = mfma4(x[r], z[r], p);
        }
        const int j = 16 * tjb + c16;
        const float bj = sBeta[j];
        float cs = 0.f, cb = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * tib + 4 * g + r;
            const float tlg = -p[r] * lg[n][r];  // dT_ij L_ij G_ij (L o G is zero on and above the diagonal)
            dm[n][r] = i > j ? -p[r] * bj * lt[n][r] : 0.f;
            const float x = xs[n][r] + bj * tlg;
            cs += x;
            cb += tlg;
            const float rs = sum_cols(x);
            if (c16 == 0) sTr[w + kW * n][4 * g + r] = rs;
        }
        cs = sum_rows(cs);
        cb = sum_rows(cb);
        if (g == 0) {
            sTc[w + kW * n][c16] = cs;
            sTb[w + kW * n][c16] = cb;
        }
    }
    __syncthreads();
    // ---- dG + dG^T for E
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        if (w + kW * n >= 10) break;
        int tib, tjb;
        lower_tile(w + kW * n, tib, tjb);
        const int j = 16 * tjb + c16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * tib + 4 * g + r;
            if (i >= j) sE[i][j] = dm[n][r];
            if (i > j) sE[j][i] = dm[n][r];
        }
    }
    // ---- decays and write rates of the chunk's tokens (the slots are complete)
    if (w == 0) {
        const int tb = lane >> 4, cc = lane & 15;
        float dg = sDp[0][lane] + sDp[1][lane] + sDh[0][lane] + sDh[1][lane];
        float db = sDb[0][lane] + sDb[1][lane];
        for (int n = 0; n < 10; ++n) {
            int tib, tjb;
            lower_tile(n, tib, tjb);
            if (tib == tb) dg += sTr[n][cc];
            if (tjb == tb) {
                dg -= sTc[n][cc];
                db += sTb[n][cc];
            }
        }
        const float z = sBeta[lane] * (sZ[0][lane] + sZ[1][lane]);
        float ds = 0.f;
        for (int n = 0; n < kW; ++n) ds += sRed[n];
        dg -= z;
        const float zt = wave_sum(z);
        if (lane == kC - 1) dg += zt + sEc[kC - 1] * ds;
        const float pre = wave_prefix_sum(dg);
        const float tot = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pre), 63));
        const float dlog = tot - pre + dg;  // sum over the chunk's tokens from this one on
        if (t0 + lane < a.L) {
            const float al = a.alpha[obase + lane];
            a.dalpha[obase + lane] = (al >= 1e-5f && al <= 1.0f) ? dlog / al : 0.f;
            a.dbeta[obase + lane] = db;
        }
    }
    __syncthreads();

    // ---- dPhi += (dG + dG^T) Phi, then q and k through the feature maps
    const bool valid = t0 + tok < a.L;
    const int64_t ko = b * a.k_sb + hk * a.k_sh + static_cast<int64_t>(t0 + (valid ? tok : 0)) * a.k_sl;
    float d1 = 0.f, d2 = 0.f;
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
        const int f0 = 16 * (2 * hb + jj) + 4 * g;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const int fb = 2 * hb + jj + 4 * hf;
            f32x4 y = dphi[jj][hf];
#pragma unroll 8
            for (int s = 0; s < 16; ++s) y = mfma4(sPhi[4 * s + g][16 * fb + c16], sE[tok][4 * s + g], y);
            dphi[jj][hf] = y;
        }
        // x/|x| of k and of k^2 (phi holds the latter over sqrt 2)
        const f32x4 p1 = ld4(&sPhi[tok][f0]), p2 = ld4(&sPhi[tok][kD + f0]), q = ld4(&sPsi[tok][f0]);
        f32x4 dq;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            d1 = fmaf(p1[r], dphi[jj][0][r], d1);
            d2 = fmaf(p2[r], dphi[jj][1][r], d2);
            dq[r] = dpsi[jj][0][r] + 2.0f * kInvSqrt2 * q[r] * dpsi[jj][1][r];
        }
        if (valid) st4_dw(a.dq + (obase + tok) * kD + f0, dq);
    }
    d1 = sum_rows(d1);
    d2 = sum_rows(d2);
    // (sDp and sDh: their readers passed the barrier above)
    if (g == 0) {
        sDp[hb][tok] = d1;
        sDh[hb][tok] = d2;
    }
    __syncthreads();
    {
        const float r1 = sR1[tok], r2 = sR2[tok];
        // the projection off x/|x|, where the norm was above eps
        const float n1 = r1 * a.feat_eps < 1.0f ? sDp[0][tok] + sDp[1][tok] : 0.f;
        const float n2 = r2 * a.feat_eps < 1.0f ? sDh[0][tok] + sDh[1][tok] : 0.f;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int f0 = 16 * (2 * hb + jj) + 4 * g;
            const f32x4 p1 = ld4(&sPhi[tok][f0]), p2 = ld4(&sPhi[tok][kD + f0]);
            f32x4 dk;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float kx = valid ? load1<DT>(a.k, ko + f0 + r) : 0.f;
                // p2 n2: both carry 1/sqrt 2 of the squares' features, (x/|x|) (g . x/|x|) has it once
                const float g1 = r1 * (dphi[jj][0][r] - p1[r] * n1);
                const float g2 = r2 * (kInvSqrt2 * dphi[jj][1][r] - 1.4142135623730951f * p2[r] * n2);
                dk[r] = g1 + 2.0f * kx * g2;
            }
            if (valid) st4_dw(a.dk + (obase + tok) * kD + f0, dk);
        }
    }
}

// Sequences are taken in groups, as many as the workspace holds.  Its full size is for two a CU
// (the chains' LDS lets two workgroups share one) and 8 GiB, at least one sequence: 2048
// sequences of 1024 tokens take 12.6 ms in groups of 512 (2.3 GB), 12.4 in one (9.2), 13.4 in
// groups of 192, 18.5 of 64; 192 of 2048 2.5 ms in one, 3.0 in two, 3.4 in three.
constexpr size_t kDeltaBwdWsCap = size_t{8} << 30;

size_t delta_backward_ws_bytes(int B, int H, int L) {
    const size_t per = seq_ws_bytes((L + kC - 1) / kC), n = static_cast<size_t>(B) * H;
    const size_t fit = std::min<size_t>(kDeltaBwdWsCap / per, 2 * static_cast<size_t>(device_cus()));
    return per * (fit < 1 ? 1 : fit < n ? fit : n);
}

template <int DT>
static hipError_t launch_group(const DeltaBwdArgs &a, int n, int NC, hipStream_t s) {
    hipError_t e;
    const dim3 block(kW * kWave);
    hipLaunchKernelGGL(delta_bwd_prep_kernel<DT>, dim3(n * NC), block, 0, s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(delta_bwd_chain_kernel<false>, dim3(n), block, 0, s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(delta_bwd_chain_kernel<true>, dim3(n), block, 0, s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(delta_bwd_grad_kernel<DT>, dim3(n * NC), block, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_delta_backward(DeltaBwdArgs a, hipStream_t stream) {
    const int NC = (a.L + kC - 1) / kC, total = a.B * a.H;
    const int group = static_cast<int>(std::min<size_t>(a.ws_bytes / seq_ws_bytes(NC), total));
    for (a.seq0 = 0; a.seq0 < total; a.seq0 += group) {
        const int n = group < total - a.seq0 ? group : total - a.seq0;
        const hipError_t e = a.dt_in == PRIME_BF16 ? launch_group<PRIME_BF16>(a, n, NC, stream)
                                                   : launch_group<PRIME_F32>(a, n, NC, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace prime
