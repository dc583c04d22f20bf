// Backward (vector-Jacobian product) of the chunked PRIME prefill on gfx950.
//
// The forward, per (sequence, head), in feature form: phi_q = [q | q*q] and
// phi_k = [k | k*k/2] (128 features each, plus a constant feature 1 on both
// sides), V' = [v | 1] (65 columns: the 65th carries the denominator), and
//   M_t = l M_{t-1} + phi_k(t) V'(t)^T        (128 x 65 plus a constant row m0 = [S0 | K0])
//   [num_t | den_t] = phi_q(t)^T M_t + m0_t,  y_t = num_t / max(den_t, eps)
// (attention.py:119-143; the chunked core of chunked_ssd.py:48-184 computes the
// same numbers).  With the output adjoint dy, let d_t = max(den_t, eps) and
//   G_t = [dy_t / d_t | -(dy_t . y_t) / d_t * [den_t >= eps]]        (65 values)
// (torch's clamp passes the gradient where den >= eps).  Then
//   dphi_q(t) = M_t G_t
//   dphi_k(j) = R_j V'(j),   dV'(j) = R_j^T phi_k(j),
//   R_j = sum_{t >= j} l^(t-j) phi_q(t) G_t^T + l^(L-1-j) dM_out,
//   dM_in = l R_0   (the adjoint of the incoming state),
// and dq = dphi_q[q] + 2 q * dphi_q[q*q], dk = dphi_k[k] + k * dphi_k[k*k/2].
//
// Two kernels, one workgroup of eight waves per sequence, 64-token chunks: four
// readout waves (16 tokens each) form a chunk's gradients while four update waves
// advance the carried state and prepare the next chunk's tiles; between two
// barriers the update waves write both to LDS (80 KB and 128 registers, so two
// workgroups share a CU).  Both passes are bound by the readout waves' chain of
// dependent products and its LDS traffic, not by HBM: 384 sequences of 2048 tokens
// take 430 us for 1.1 GB (572 with four waves that did everything in turn and
// waited for each prefetched row where it was loaded); 768 of 256, 97 (139).
//
//  * dq pass (chunks in order).  The forward chunk loop again -- the value
//    columns of M carried in MFMA accumulators, a bf16 copy of them in LDS for
//    the readout -- and per chunk: scores S^T, num = A v + pin (phi_q M + S0),
//    G, then P = mask * (G V'^T) and dphi_q = P phi_k + pin G M^T.  The
//    denominator is formed in fp32 (row sums of the masked scores, and the K
//    column of M kept in fp32 on the VALU): whether the clamp is active
//    switches the gradient, so that decision must not rest on bf16 operands.
//    It writes dq and, per token, 1/d and the denominator adjoint (8 bytes)
//    for the second pass.
//  * dk, dv pass (chunks in reverse).  The dual state W (128 x 65 plus a
//    constant row W1) carries sum_{t >= e} l^(t-e+1) phi_q(t) G_t^T + l^(L-e) dM_out
//    for the chunk end e; per chunk A = mask * (1 + phi_q phi_k^T) and
//    P = mask * (G V'^T) give dV' = A^T G + l^(e-1-j) (W^T phi_k + W1) and
//    dphi_k = P^T phi_q + l^(e-1-j) W V', then W <- l^n W + sum l^(t-c0+1) phi_q G^T.
//    After chunk 0, W is the incoming state's adjoint.
//
// MFMA operand conventions are those of the forward kernels: an operand whose
// K index runs along an LDS row is read with row_op; one whose K index runs
// down a column (tokens, or value columns of a transposed copy) with tr_op,
// whose lane holds K slots {32ks + 4g + t, 32ks + 16 + 4g + t}; accumulators
// of a transposed block S^T[j][i] (lane: rows 16jb + 4g + r, column i) are an
// A operand for row i with that same K permutation.  Every MFMA runs under
// wave-uniform control flow.

#include <algorithm>

#include "prefill_common.h"

namespace prime {
namespace {

constexpr int kPV = kD + 16;   // pitch of 80-wide rows ([v | 0..], [g | gden | 0..])
constexpr int kSR = kD + 1;    // rows of a transposed state copy: 64 value columns + the K column

__device__ __forceinline__ void st16(uint16_t *p, u32x4 x) { *reinterpret_cast<u32x4 *>(p) = x; }

// 8 consecutive elements of a row of dtype dt as loaded (16 bytes, or two times
// 16 for fp32), as packed bf16 (round to nearest even)
__device__ __forceinline__ u32x4 pack_raw(const u32x4 (&x)[2], int dt) {
    if (dt == PRIME_BF16) return x[0];
    float f[8];
    if (dt == PRIME_F32) {
        const f32x4 lo = __builtin_bit_cast(f32x4, x[0]), hi = __builtin_bit_cast(f32x4, x[1]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[i] = lo[i];
            f[4 + i] = hi[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = h16_bits_to_f32(static_cast<uint16_t>(x[0][i] & 0xFFFFu));
            f[2 * i + 1] = h16_bits_to_f32(static_cast<uint16_t>(x[0][i] >> 16));
        }
    }
    return pack8(f);
}

__device__ __forceinline__ u32x4 and4(u32x4 x, uint32_t m) { return u32x4{x[0] & m, x[1] & m, x[2] & m, x[3] & m}; }

// s * x * x of 8 packed bf16, repacked
__device__ __forceinline__ u32x4 sq8(u32x4 x, float s) {
    float f[8];
    unpack8(x, f);
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = pack2(s * f[2 * i] * f[2 * i], s * f[2 * i + 1] * f[2 * i + 1]);
    return r;
}

// 8 floats times s, packed to bf16
__device__ __forceinline__ u32x4 pack8s(const float (&f)[8], float s) {
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = pack2(s * f[2 * i], s * f[2 * i + 1]);
    return r;
}

// A operand from two transposed accumulator blocks (K slots 0..3 and 4..7)
__device__ __forceinline__ bf16x8 acc_op(const f32x4 &lo, const f32x4 &hi) {
    return as_bf16x8(u32x4{pack2(lo[0], lo[1]), pack2(lo[2], lo[3]), pack2(hi[0], hi[1]), pack2(hi[2], hi[3])});
}

// A operand of one row with the tr_op K permutation: elements [32ks + 4g, +4)
// and [32ks + 16 + 4g, +4) of the row, times s
__device__ __forceinline__ bf16x8 perm_row_op(const uint16_t *row, int ks, int g, float s) {
    const uint2 a = *reinterpret_cast<const uint2 *>(row + 32 * ks + 4 * g);
    const uint2 b = *reinterpret_cast<const uint2 *>(row + 32 * ks + 16 + 4 * g);
    const uint32_t w[4] = {a.x, a.y, b.x, b.y};
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        r[i] = pack2(s * __uint_as_float(w[i] << 16), s * __uint_as_float(w[i] & 0xFFFF0000u));
    return as_bf16x8(r);
}

// an operand's 8 bf16 values times per-slot weights, repacked
__device__ __forceinline__ bf16x8 scale_op(bf16x8 x, const float (&wt)[8]) {
    const u32x4 r = __builtin_bit_cast(u32x4, x);
    float f[8];
    unpack8(r, f);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] *= wt[i];
    return as_bf16x8(pack8(f));
}

// v[fb][r] to base[o + 16 fb + r] (o includes the lane's 4g), in dtype dt: one
// 16- or 8-byte store per block where the rows allow it (vec)
__device__ __forceinline__ void store_row16(void *base, int dt, bool vec, int64_t o, const f32x4 (&v)[4]) {
    if (dt == PRIME_F32) {
        float *p = static_cast<float *>(base) + o;
#pragma unroll
        for (int fb = 0; fb < 4; ++fb) {
            if (vec) {
                *reinterpret_cast<f32x4 *>(p + 16 * fb) = v[fb];
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) p[16 * fb + r] = v[fb][r];
            }
        }
    } else {
        uint16_t *p = static_cast<uint16_t *>(base) + o;
#pragma unroll
        for (int fb = 0; fb < 4; ++fb) {
            uint2 x;
            if (dt == PRIME_BF16) {
                x = uint2{pack2(v[fb][0], v[fb][1]), pack2(v[fb][2], v[fb][3])};
            } else {
                uint32_t hb[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) hb[r] = f32_to_h16_bits(v[fb][r]);
                x = uint2{hb[0] | hb[1] << 16, hb[2] | hb[3] << 16};
            }
            if (vec) {
                *reinterpret_cast<uint2 *>(p + 16 * fb) = x;
            } else {
                p[16 * fb] = static_cast<uint16_t>(x.x);
                p[16 * fb + 1] = static_cast<uint16_t>(x.x >> 16);
                p[16 * fb + 2] = static_cast<uint16_t>(x.y);
                p[16 * fb + 3] = static_cast<uint16_t>(x.y >> 16);
            }
        }
    }
}

// four consecutive packed bf16 at p (8-byte aligned)
__device__ __forceinline__ f32x4 unpack4(const uint16_t *p) {
    const uint2 x = *reinterpret_cast<const uint2 *>(p);
    return f32x4{__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xFFFF0000u), __uint_as_float(x.y << 16),
                 __uint_as_float(x.y & 0xFFFF0000u)};
}

// an operand row with the tr_op K permutation, as it lies in LDS
__device__ __forceinline__ bf16x8 perm_row(const uint16_t *row, int ks, int g) {
    const uint2 a = *reinterpret_cast<const uint2 *>(row + 32 * ks + 4 * g);
    const uint2 b = *reinterpret_cast<const uint2 *>(row + 32 * ks + 16 + 4 * g);
    return as_bf16x8(u32x4{a.x, a.y, b.x, b.y});
}

// Keeps a value's computation before this point (an update wave prepares the next
// tiles before the barrier that the readout waves are still on their way to).
__device__ __forceinline__ void settle(u32x4 &x) { asm volatile("" : "+v"(x)); }

// Orders a wave's LDS writes before its own later LDS reads by other lanes.
__device__ __forceinline__ void lds_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// An index the compiler cannot trace: addresses formed from it are formed where
// they are used instead of being kept in registers over the whole chunk loop.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// One chunk's inputs for one update thread: rows ra and ra + 32, columns
// col..col+7, as they lie in memory (q, k, v are bf16 here; dy of any dtype).
// Nothing may touch the results before they are needed, or the wave waits out
// the latency where the load is issued.  q, k and v are loaded a chunk ahead; dy
// and its two per-token numbers only once the state update is done (the readout
// waves take longer), so that the loads in flight and the state fit 128 registers.
struct Rows {
    u32x4 q[2], k[2], v[2], dy[2][2];
    float inv[2], gden[2];
};

template <bool KV>
__device__ __forceinline__ void load_qkv(Rows &R, const BwdArgs &a, int b, int h, int c, int ra, int col) {
    const int64_t t0 = static_cast<int64_t>(c) * kC;
    const int last = min(kC, a.L - c * kC) - 1;
    const uint16_t *q = static_cast<const uint16_t *>(a.q) + b * a.q_sb + h * a.q_sh + t0 * a.q_sl;
    const uint16_t *k = static_cast<const uint16_t *>(a.k) + b * a.k_sb + h * a.k_sh + t0 * a.k_sl;
    const uint16_t *v = static_cast<const uint16_t *>(a.v) + b * a.v_sb + h * a.v_sh + t0 * a.v_sl;
    ra = opaque(ra);  // scalar bases plus a lane offset formed here
    col = opaque(col);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int64_t t = min(ra + 32 * s, last);  // clamped; rows past L are zeroed when prepared
        R.q[s] = *reinterpret_cast<const u32x4 *>(q + t * a.q_sl + col);
        if constexpr (KV) {
            R.k[s] = *reinterpret_cast<const u32x4 *>(k + t * a.k_sl + col);
            R.v[s] = *reinterpret_cast<const u32x4 *>(v + t * a.v_sl + col);
        }
    }
}

template <bool DEN>
__device__ __forceinline__ void load_dy(Rows &R, const BwdArgs &a, int b, int h, int c, int ra, int col) {
    const int64_t t0 = static_cast<int64_t>(c) * kC;
    const int last = min(kC, a.L - c * kC) - 1;
    const int es = a.dt_dy == PRIME_F32 ? 4 : 2, step = a.dt_dy == PRIME_F32 ? 16 : 0;
    const char *dy = static_cast<const char *>(a.dy) + es * (b * a.dy_sb + h * a.dy_sh + t0 * a.dy_sl);
    const size_t o = static_cast<size_t>(b * a.H + h) * a.L + t0;
    ra = opaque(ra);
    col = opaque(col);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int64_t t = min(ra + 32 * s, last);
        const char *p = dy + es * (t * a.dy_sl + col);
        R.dy[s][0] = *reinterpret_cast<const u32x4 *>(p);
        R.dy[s][1] = *reinterpret_cast<const u32x4 *>(p + step);
        if constexpr (DEN) {
            R.inv[s] = a.inv_den[o + t];
            R.gden[s] = a.g_den[o + t];
        }
    }
}

}  // namespace

// ---------------------------------------------------------------- dq pass
// DIN: the dense double clamp with an incoming state (BwdArgs::dense_in)
template <bool DIN>
__global__ __launch_bounds__(512, DIN ? 2 : 4) void prefill_bwd_dq_kernel(const BwdArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t sQf[kC][kPT];   // [q | q*q]
    __shared__ __attribute__((aligned(16))) uint16_t sKf[kC][kPT];   // [k | k*k/2]
    __shared__ __attribute__((aligned(16))) uint16_t sV[kC][kPV];    // v
    __shared__ __attribute__((aligned(16))) uint16_t sG[kC][kPV];    // dy
    __shared__ __attribute__((aligned(16))) uint16_t sSt[kD][kPT];   // bf16 value columns of M^T entering the chunk
    // fp32: the K column of M (the denominator's moments) entering the chunk, S0, K0
    __shared__ __attribute__((aligned(16))) float sKv[kF], sS0[kD];
    __shared__ float sK0[1], sPw[kC + 2], sPs[kC + 2];
    __shared__ float sRedK[kF];  // the chunk's K increment (written and read by the same update wave)
    // dense double clamp with an incoming state: the incoming [K1; K2/2] and K0
    // (the carried K above is then the call's own), and per token of the chunk
    // l^(t+1) times the part of the outer-clamp denominator adjoint that the
    // inner clamp withholds from the call's tokens (sDh)
    __shared__ __attribute__((aligned(16))) float sKin[kF];
    __shared__ float sK0in[1], sDh[kC];
    // the state-update weights l^(n-1-j) of a full chunk (0) and of the
    // sequence's last chunk (1, n = its valid tokens), and the same weights split
    // into three bf16 parts (hi, mid, lo: about fp32 precision in sum), row 3
    // zero: an MFMA operand whose columns (or rows) 0..2 are the parts
    __shared__ __attribute__((aligned(16))) float sWt[2][kC];
    __shared__ __attribute__((aligned(16))) uint16_t sWp[2][4][kC];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const bool is_u = wave >= 4;                // update role
    const int w = wave & 3, ut = tid & 255;     // wave and thread index within the role
    const int g = lane >> 4, c16 = lane & 15;
    const int tr_r = c16 >> 2, tr_c = 4 * (c16 & 3);
    const int unit = blockIdx.x;
    if (unit >= a.B * a.H * a.G) return;
    const int seq = unit / a.G, seg = unit - seq * a.G;
    const int b = seq / a.H, h = seq - b * a.H;
    const float lam = a.decay[h];
    const int NC = (a.L + kC - 1) / kC;
    const int c_begin = seg * a.cps, c_end = min(c_begin + a.cps, NC);
    // the state entering the first chunk: state_in, or the segment's slot (same components)
    const float *S0p, *S1p, *S2p, *K0p, *K1p, *K2p;
    if (a.G > 1) {
        const float *slot = a.ws + static_cast<size_t>(unit) * kWsStride;
        S1p = slot + kWsS1; S2p = slot + kWsS2; S0p = slot + kWsS0;
        K1p = slot + kWsK1; K2p = slot + kWsK2; K0p = slot + kWsK0;
    } else if (a.s1i) {
        S1p = a.s1i + static_cast<size_t>(seq) * kD * kD; S2p = a.s2i + static_cast<size_t>(seq) * kD * kD;
        S0p = a.s0i + static_cast<size_t>(seq) * kD; K1p = a.k1i + static_cast<size_t>(seq) * kD;
        K2p = a.k2i + static_cast<size_t>(seq) * kD; K0p = a.k0i + seq;
    } else {
        S0p = S1p = S2p = K0p = K1p = K2p = nullptr;
    }

    if (tid < kC + 2) {
        const PowSum t = pow_sum(lam, tid);
        sPw[tid] = static_cast<float>(t.p);
        sPs[tid] = static_cast<float>(t.s);
    }
    constexpr bool din = DIN;  // (then G == 1: the S*p are state_in)

    __syncthreads();  // power tables
    if (tid < 2 * kC) {  // the two weight tables (read after the chunk loop's first barrier)
        const int t = tid & (kC - 1), which = tid >> 6;
        const int nv = which ? a.L - (NC - 1) * kC : kC;
        const float wv = t < nv ? sPw[nv - 1 - t] : 0.f;
        sWt[which][t] = wv;
        const uint16_t hi = f32_to_bf16_bits(wv);
        const float r1 = wv - bf16_bits_to_f32(hi);
        const uint16_t mid = f32_to_bf16_bits(r1);
        sWp[which][0][t] = hi;
        sWp[which][1][t] = mid;
        sWp[which][2][t] = f32_to_bf16_bits(r1 - bf16_bits_to_f32(mid));
        sWp[which][3][t] = 0u;
    }
    if (is_u) {
        // ================ update role: the carried state and the tiles
        // value columns of M (features 32w..32w+31 of this wave, value blocks 0..3) from state_in
        f32x4 st[2][4];
        // the denominator's moments [K1; K2/2] in fp32, feature 32w + lane (lane < 32);
        // S0 of value column 16w + c16 (lane group 0); K0
        float kv = 0.f, s0 = 0.f, k0 = 0.f;
#pragma unroll
        for (int fi = 0; fi < 2; ++fi)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) st[fi][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (S1p) {
            const float *Sp = w < 2 ? S1p : S2p, *Kp = w < 2 ? K1p : K2p;  // waves 0, 1 hold features 0..63
            const float sc = w < 2 ? 1.0f : 0.5f;
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int fr = (16 * (2 * w + fi) + 4 * g + r) & (kD - 1);
                        st[fi][nb][r] = Sp[fr * kD + 16 * nb + c16];
                    }
            kv = sc * Kp[(32 * w + (lane & 31)) & (kD - 1)];
            s0 = S0p[16 * w + c16];
            k0 = K0p[0];
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) st[fi][nb] *= sc;
        }
        if (din) {
            if (lane < 32) sKin[32 * w + lane] = kv;
            if (ut == 0) sK0in[0] = k0;
            kv = k0 = 0.f;
        }
        float corr = 0.f;  // (din) this thread's feature (ut < 128) or K0 (ut == 128) of the correction
        const int ra = ut >> 3, col = 8 * (ut & 7);
        Rows R;
        u32x4 q2[2], k2[2], gr[2];  // squares, and dy as bf16
        auto prepare = [&](int c) {
            const int nv = min(kC, a.L - c * kC);
            load_dy<false>(R, a, b, h, c, ra, col);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (nv < kC) {
                    const uint32_t m = ra + 32 * s < nv ? 0xFFFFFFFFu : 0u;
                    R.q[s] = and4(R.q[s], m);
                    R.k[s] = and4(R.k[s], m);
                    R.v[s] = and4(R.v[s], m);
                }
                q2[s] = sq8(R.q[s], 1.f);
                k2[s] = sq8(R.k[s], 0.5f);
                settle(q2[s]);
                settle(k2[s]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                gr[s] = pack_raw(R.dy[s], a.dt_dy);
                if (nv < kC) gr[s] = and4(gr[s], ra + 32 * s < nv ? 0xFFFFFFFFu : 0u);
                settle(gr[s]);
            }
        };
        auto publish = [&]() {  // the prepared tiles and the state entering their chunk
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int row = ra + 32 * s;
                st16(&sQf[row][col], R.q[s]);
                st16(&sQf[row][kD + col], q2[s]);
                st16(&sKf[row][col], R.k[s]);
                st16(&sKf[row][kD + col], k2[s]);
                st16(&sV[row][col], R.v[s]);
                st16(&sG[row][col], gr[s]);
            }
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb)
                    *reinterpret_cast<uint2 *>(&sSt[16 * nb + c16][16 * (2 * w + fi) + 4 * g]) =
                        uint2{pack2(st[fi][nb][0], st[fi][nb][1]), pack2(st[fi][nb][2], st[fi][nb][3])};
            if (lane < 32) sKv[32 * w + lane] = kv;
            if (g == 0) sS0[16 * w + c16] = s0;
            if (ut == 0) sK0[0] = k0;
        };
        load_qkv<true>(R, a, b, h, c_begin, ra, col);
        prepare(c_begin);
        publish();
        if (c_begin + 1 < c_end) load_qkv<true>(R, a, b, h, c_begin + 1, ra, col);
        for (int c = c_begin; c < c_end; ++c) {
            const int nvalid = min(kC, a.L - c * kC);
            const int wsel = nvalid == kC ? 0 : 1;  // weights of a full chunk or of the last one
            __syncthreads();  // tiles of chunk c and M_c in LDS
            if (c + 1 < c_end) {
                // ---- M <- l^n M + (w phi_k)^T v with w_j = l^(n-1-j) on the A operand's
                // token slots; S0 and K = [K1; K2/2] (fp32) as partial sums over all threads
                const float ln = sPw[nvalid];
#pragma unroll
                for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
                        for (int r = 0; r < 4; ++r) st[fi][nb][r] *= ln;
                // K and S0 increments on MFMA, against the three parts of w (fp32-accurate
                // sums: K decides the clamp): dk[fi] rows = features, columns 0..2 = parts;
                // ds0 rows 0..2 = parts, columns = value block w
                f32x4 dk[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
                f32x4 ds0 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    float wt[8];
                    {
                        const f32x4 w0 = *reinterpret_cast<const f32x4 *>(&sWt[wsel][32 * ks + 4 * g]);
                        const f32x4 w1 = *reinterpret_cast<const f32x4 *>(&sWt[wsel][32 * ks + 16 + 4 * g]);
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            wt[t] = w0[t];
                            wt[4 + t] = w1[t];
                        }
                    }
                    // lane (g, c16): part min(c16, 3) of w at its eight token slots, the
                    // same slots as the transposed operands (token 32ks + 16(t/4) + 4g + t%4)
                    const int pr = min(c16, 3);
                    const uint2 p0 = *reinterpret_cast<const uint2 *>(&sWp[wsel][pr][32 * ks + 4 * g]);
                    const uint2 p1 = *reinterpret_cast<const uint2 *>(&sWp[wsel][pr][32 * ks + 16 + 4 * g]);
                    const bf16x8 wpart = as_bf16x8(u32x4{p0.x, p0.y, p1.x, p1.y});
                    bf16x8 ak[2];
#pragma unroll
                    for (int fi = 0; fi < 2; ++fi) {
                        const uint16_t *pk = &sKf[32 * ks + 4 * g + tr_r][16 * (2 * w + fi) + tr_c];
                        const bf16x8 raw = tr_op<false>(pk, pk + 16 * kPT, 0).h;
                        dk[fi] = mfma(raw, wpart, dk[fi]);
                        ak[fi] = scale_op(raw, wt);
                    }
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb) {
                        const uint16_t *p0v = &sV[32 * ks + 4 * g + tr_r][16 * nb + tr_c];
                        const bf16x8 vb = tr_op<false>(p0v, p0v + 16 * kPV, 0).h;
#pragma unroll
                        for (int fi = 0; fi < 2; ++fi) st[fi][nb] = mfma(ak[fi], vb, st[fi][nb]);
                        if (nb == w) ds0 = mfma(wpart, vb, ds0);  // wave-uniform
                    }
                }
                {
                    // K increment of features 16(2w + fi) + 4g + r: the quad (columns 0..3) sum
#pragma unroll
                    for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            float x = dk[fi][r];
                            x += xor_lane<1>(x);
                            x += xor_lane<2>(x);
                            if (c16 == 0) sRedK[16 * (2 * w + fi) + 4 * g + r] = x;
                        }
                    // S0 of value column 16w + c16: rows 0..2 of the increment (lane group g = 0)
                    s0 = ln * s0 + ((ds0[0] + ds0[1]) + ds0[2]);
                    k0 = ln * k0 + sPs[nvalid];
                    lds_wave_sync();
                    if (lane < 32) kv = ln * kv + sRedK[32 * w + lane];
                }
                __builtin_amdgcn_sched_barrier(0);
                prepare(c + 1);
            }
            __syncthreads();  // every read of chunk c's tiles and of M_c is done
            if (din) {  // correction: sum over the chunk of sDh_t phi_q(t) (chunk c's tiles are still in LDS)
                if (ut < kF) {
                    float sacc = 0.f;
                    for (int i = 0; i < nvalid; ++i) sacc += sDh[i] * bf16_bits_to_f32(sQf[i][ut]);
                    corr += sacc;
                } else if (ut == kF) {
                    float sacc = 0.f;
                    for (int i = 0; i < nvalid; ++i) sacc += sDh[i];
                    corr += sacc;
                }
                __syncthreads();  // before the tiles change
            }
            if (c + 1 < c_end) {
                publish();
                __builtin_amdgcn_sched_barrier(0);
                if (c + 2 < c_end) load_qkv<true>(R, a, b, h, c + 2, ra, col);
            }
        }
        if (din && ut <= kF) a.kcorr[static_cast<size_t>(seq) * kBwdCorr + ut] = corr;
        return;
    }

    // ================ readout role: dq of rows 16w..16w+15 of every chunk
    // Every product is formed transposed (tokens on the columns), so a lane holds
    // one token, iw, and four consecutive columns of each 16-wide block: G becomes
    // an operand in registers, per-token factors are lane scalars, and rows are
    // stored 8 or 16 bytes at a time.  (powers from the table: sPw[n] is l^n
    // rounded from fp64)
    const int iw = 16 * w + c16;
    float mask[4][4];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = iw - (16 * jb + 4 * g + r);
            mask[jb][r] = (jb <= w && d >= 0) ? sPw[max(d, 0)] : 0.f;
        }
    const float pinc = sPw[iw + 1];
    for (int c = c_begin; c < c_end; ++c) {
        const int nvalid = min(kC, a.L - c * kC);
        // (din) l^(64 c): the incoming state's decay to the chunk's start
        const float lc = din ? static_cast<float>(int_pow(lam, int64_t{kC} * c)) : 0.f;
        __syncthreads();  // tiles of chunk c and M_c in LDS
        // ---- scores S^T[j][iw] (blocks jb <= w), masked: A = l^(i-j) (1 + phi_q . phi_k)
        f32x4 sT[4];
#pragma unroll
        for (int jb = 0; jb < 4; ++jb) {
            sT[jb] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (jb > w) continue;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                sT[jb] = mfma(as_bf16x8(lds128(&sKf[16 * jb + c16][32 * ks + 8 * g])),
                              as_bf16x8(lds128(&sQf[iw][32 * ks + 8 * g])), sT[jb]);
#pragma unroll
            for (int r = 0; r < 4; ++r) sT[jb][r] = mask[jb][r] * (1.0f + sT[jb][r]);
        }
        // ---- numerator of row iw, columns 16nb + 4g + r: A V + pin (phi_q M + S0)
        f32x4 acc[4], accC[4];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[nb] = accC[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            if (2 * ks > w) continue;
            const bf16x8 A = acc_op(sT[2 * ks], sT[2 * ks + 1]);
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
                const uint16_t *p0 = &sV[32 * ks + 4 * g + tr_r][16 * nb + tr_c];
                acc[nb] = mfma(tr_op<false>(p0, p0 + 16 * kPV, 0).h, A, acc[nb]);
            }
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const bf16x8 Aq = as_bf16x8(lds128(&sQf[iw][32 * ks + 8 * g]));
#pragma unroll
            for (int nb = 0; nb < 4; ++nb)
                accC[nb] = mfma(as_bf16x8(lds128(&sSt[16 * nb + c16][32 * ks + 8 * g])), Aq, accC[nb]);
        }
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const f32x4 m0 = *reinterpret_cast<const f32x4 *>(&sS0[16 * nb + 4 * g]);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[nb][r] += pinc * (accC[nb][r] + m0[r]);
        }
        // ---- denominator of row iw in fp32 (whether the clamp is active decides
        // the gradient): row sum of the masked scores + pin (phi_q . K + K0)
        float dsum = 0.f, dcar = 0.f, dcin = 0.f;
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
#pragma unroll
            for (int r = 0; r < 4; ++r) dsum += sT[jb][r];
#pragma unroll
        for (int t = 0; t < 4; ++t) {  // features 32g + 8t + 0..7 of row iw, one 16-byte read
            float qf[8];
            unpack8(lds128(&sQf[iw][((32 * g) & (kD - 1)) + 8 * t]), qf);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float ph = g < 2 ? qf[e] : qf[e] * qf[e];
                dcar += ph * sKv[32 * g + 8 * t + e];
                if (din) dcin += ph * sKin[32 * g + 8 * t + e];
            }
        }
        dsum = sum_lane32(sum_lane16(dsum));
        dcar = sum_lane32(sum_lane16(dcar));
        const float den = dsum + pinc * (dcar + sK0[0]);
        // single clamp max(den, eps), or (din) the double clamp max(max(den, eps) + cr, eps) with the
        // incoming state's denominator term cr = l^(t+1) (K0 + phi_q . K) outside the inner clamp
        const float d1 =
            din ? fmaxf(den, a.eps) + lc * pinc * (sum_lane32(sum_lane16(dcin)) + sK0in[0]) : den;
        const float inv = 1.0f / fmaxf(d1, a.eps);
        // ---- G of row iw, columns 16nb + 4g + r; gop: its bf16 values as an operand in the tr_op K order
        const bool valid = iw < nvalid;
        float part = 0.f;
        f32x4 gn[4];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const f32x4 dyv = unpack4(&sG[iw][16 * nb + 4 * g]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                part += dyv[r] * (acc[nb][r] * inv);
                gn[nb][r] = valid ? dyv[r] * inv : 0.f;
            }
        }
        part = sum_lane32(sum_lane16(part));
        // the outer clamp's adjoint, and the call's share of it (inner clamp)
        const float gout = (valid && d1 >= a.eps) ? -part * inv : 0.f;
        const float gden = den >= a.eps ? gout : 0.f;
        if (din && g == 0) sDh[iw] = lc * pinc * (gout - gden);
        const bf16x8 gop[2] = {acc_op(gn[0], gn[1]), acc_op(gn[2], gn[3])};
        // ---- P^T[j][iw] = mask * (v_j . g_iw + gden)
        f32x4 pT[4];
#pragma unroll
        for (int jb = 0; jb < 4; ++jb) {
            pT[jb] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (jb > w) continue;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) pT[jb] = mfma(perm_row(&sV[16 * jb + c16][0], ks, g), gop[ks], pT[jb]);
#pragma unroll
            for (int r = 0; r < 4; ++r) pT[jb][r] = mask[jb][r] * (pT[jb][r] + gden);
        }
        // ---- dphi_q of row iw, features 16fb + 4g + r: P phi_k + pin G M^T
        f32x4 dphi[8];
#pragma unroll
        for (int fb = 0; fb < 8; ++fb) dphi[fb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            if (2 * ks > w) continue;
            const bf16x8 A = acc_op(pT[2 * ks], pT[2 * ks + 1]);
#pragma unroll
            for (int fb = 0; fb < 8; ++fb) {
                const uint16_t *p0 = &sKf[32 * ks + 4 * g + tr_r][16 * fb + tr_c];
                dphi[fb] = mfma(tr_op<false>(p0, p0 + 16 * kPT, 0).h, A, dphi[fb]);
            }
        }
        const float pin8[8] = {pinc, pinc, pinc, pinc, pinc, pinc, pinc, pinc};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const bf16x8 A = scale_op(gop[ks], pin8);
#pragma unroll
            for (int fb = 0; fb < 8; ++fb) {
                const uint16_t *p0 = &sSt[32 * ks + 4 * g + tr_r][16 * fb + tr_c];
                dphi[fb] = mfma(tr_op<false>(p0, p0 + 16 * kPT, 0).h, A, dphi[fb]);
            }
        }
#pragma unroll
        for (int fb = 0; fb < 8; ++fb) {  // the denominator: K column of M, and (din) the incoming K under the outer clamp
            const f32x4 kf = *reinterpret_cast<const f32x4 *>(&sKv[16 * fb + 4 * g]);
#pragma unroll
            for (int r = 0; r < 4; ++r) dphi[fb][r] += (pinc * gden) * kf[r];
            if (din) {
                const f32x4 ki = *reinterpret_cast<const f32x4 *>(&sKin[16 * fb + 4 * g]);
#pragma unroll
                for (int r = 0; r < 4; ++r) dphi[fb][r] += (lc * pinc * gout) * ki[r];
            }
        }
        // ---- dq = dphi[q] + 2 q dphi[q*q]
        if (valid) {
            f32x4 dv[4];
#pragma unroll
            for (int fb = 0; fb < 4; ++fb) {
                const f32x4 qv = unpack4(&sQf[iw][16 * fb + 4 * g]);
#pragma unroll
                for (int r = 0; r < 4; ++r) dv[fb][r] = dphi[fb][r] + 2.0f * qv[r] * dphi[fb + 4][r];
            }
            const int64_t i = c * kC + opaque(iw);
            store_row16(a.dq, a.dt_g, a.g_vec, b * a.g_sb + h * a.g_sh + i * a.g_sl + 4 * g, dv);
            // 1/d and the denominator adjoint: even lane groups the one, odd the other
            (g & 1 ? a.g_den : a.inv_den)[static_cast<size_t>(seq) * a.L + i] = g & 1 ? gden : inv;
        }
        __syncthreads();  // every read of chunk c's tiles and of M_c is done
        if (din) __syncthreads();  // (the correction's reads too)
    }
}

// ---------------------------------------------------------------- dk, dv pass
// DUAL: the dual-state pass of a segment only -- from zero, no dk / dv, the
// segment's contribution sum_t l^(t-s0+1) phi_q(t) G_t^T written to its slot.
template <bool DUAL>
__global__ __launch_bounds__(DUAL ? 256 : 512, DUAL ? 2 : 4) void prefill_bwd_dkv_kernel(const BwdArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t sQf[kC][kPT];   // [q | q*q]
    __shared__ __attribute__((aligned(16))) uint16_t sKf[kC][kPT];   // [k | k*k/2]
    __shared__ __attribute__((aligned(16))) uint16_t sV[kC][kPV];    // [v | 0..]
    __shared__ __attribute__((aligned(16))) uint16_t sG[kC][kPV];    // [dy / d | gden | 0..]
    __shared__ __attribute__((aligned(16))) uint16_t sW[kSR][kPT];   // bf16 W^T at the chunk end
    __shared__ __attribute__((aligned(16))) float sW1[kSR], sGd[kC];
    __shared__ float sPw[kC + 2];
    __shared__ __attribute__((aligned(16))) float sOm[kC];  // om_t = l^(t+1) (= sPw[t + 1]), 16-byte aligned
    // om_t = l^(t+1) split into three bf16 parts (hi, mid, lo), row 3 zero: the
    // A operand of the W1 increment on MFMA
    __shared__ __attribute__((aligned(16))) uint16_t sOmp[4][kC];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const bool is_u = DUAL || wave >= 4;     // update role
    const int w = wave & 3, ut = tid & 255;  // wave and thread index within the role
    const int g = lane >> 4, c16 = lane & 15;
    const int tr_r = c16 >> 2, tr_c = 4 * (c16 & 3);
    const int unit = blockIdx.x;
    if (unit >= a.B * a.H * a.G) return;
    const int seq = unit / a.G, seg = unit - seq * a.G;
    const int b = seq / a.H, h = seq - b * a.H;
    const float lam = a.decay[h];
    const int NC = (a.L + kC - 1) / kC;
    const int c_begin = seg * a.cps, c_end = min(c_begin + a.cps, NC);
    const size_t so1 = static_cast<size_t>(seq) * kD * kD, so0 = static_cast<size_t>(seq) * kD;
    float *slot = a.G > 1 ? a.ws + static_cast<size_t>(unit) * kWsStride : nullptr;

    if (tid < kC + 2) sPw[tid] = static_cast<float>(pow_sum(lam, tid).p);
    if (tid < kC) {
        const float om = static_cast<float>(pow_sum(lam, tid + 1).p);
        sOm[tid] = om;
        const uint16_t hi = f32_to_bf16_bits(om);
        const float r1 = om - bf16_bits_to_f32(hi);
        const uint16_t mid = f32_to_bf16_bits(r1);
        sOmp[0][tid] = hi;
        sOmp[1][tid] = mid;
        sOmp[2][tid] = f32_to_bf16_bits(r1 - bf16_bits_to_f32(mid));
        sOmp[3][tid] = 0u;
    }
    for (int idx = tid; idx < kC * 16; idx += DUAL ? 256 : 512) {
        const int row = idx >> 4, cc = kD + (idx & 15);
        sV[row][cc] = 0u;
        sG[row][cc] = 0u;
    }

    __syncthreads();  // power table

    if (is_u) {
        // ================ update role: the dual state and the tiles
        // dual state W (features 32w..32w+31, value blocks 0..4) from the final
        // state's adjoint or the segment's slot (W at its end, in this kernel's
        // convention): one uniform choice of source, then every load in flight at once
        const float *W1p = nullptr, *W2p = nullptr, *W0p = nullptr, *Wk1p = nullptr, *Wk2p = nullptr, *Wk0p = nullptr;
        float two = 1.0f;  // rows 64.. of M hold S2/2 and K2/2
        if (!DUAL && slot) {
            W1p = slot + kWsS1; W2p = slot + kWsS2; W0p = slot + kWsS0;
            Wk1p = slot + kWsK1; Wk2p = slot + kWsK2; Wk0p = slot + kWsK0;
        } else if (!DUAL && a.ds1o) {
            W1p = a.ds1o + so1; W2p = a.ds2o + so1; W0p = a.ds0o + so0;
            Wk1p = a.dk1o + so0; Wk2p = a.dk2o + so0; Wk0p = a.dk0o + seq;
            two = 2.0f;
        }
        f32x4 st[2][5];
#pragma unroll
        for (int fi = 0; fi < 2; ++fi)
#pragma unroll
            for (int nb = 0; nb < 5; ++nb) st[fi][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
        // constant row of W: column 16w + c16 (lane group 0), and the gden column
        float w1 = 0.f, w1g = 0.f;
        if (W1p) {
            const float *Wp = w < 2 ? W1p : W2p, *Wk = w < 2 ? Wk1p : Wk2p;  // waves 0, 1 hold features 0..63
            const float sc = w < 2 ? 1.0f : two;
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 5; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int fr = (16 * (2 * w + fi) + 4 * g + r) & (kD - 1);
                        st[fi][nb][r] = nb < 4 ? Wp[fr * kD + 16 * nb + c16] : Wk[fr];
                    }
            w1 = W0p[16 * w + c16];
            w1g = Wk0p[0];
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 5; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) st[fi][nb][r] = nb < 4 || c16 == 0 ? sc * st[fi][nb][r] : 0.f;
        }
        const int ra = ut >> 3, col = 8 * (ut & 7);
        Rows R;
        u32x4 gr[2];  // dy / d as bf16
        float gdr[2];
        auto prepare = [&](int c) {
            const int nv = min(kC, a.L - c * kC);
            load_dy<true>(R, a, b, h, c, ra, col);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const bool ok = ra + 32 * s < nv;
                gdr[s] = ok ? R.gden[s] : 0.f;
                float gn[8];
                unpack8(pack_raw(R.dy[s], a.dt_dy), gn);
                gr[s] = pack8s(gn, ok ? R.inv[s] : 0.f);
                settle(gr[s]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (nv < kC) {
                    const uint32_t m = ra + 32 * s < nv ? 0xFFFFFFFFu : 0u;
                    R.q[s] = and4(R.q[s], m);
                    if constexpr (!DUAL) {
                        R.k[s] = and4(R.k[s], m);
                        R.v[s] = and4(R.v[s], m);
                    }
                }
            }
        };
        auto publish = [&]() {  // the prepared tiles and W at their chunk's end
            const int t = opaque(ut), ra = t >> 3, col = 8 * (t & 7);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int row = ra + 32 * s;
                st16(&sQf[row][col], R.q[s]);
                st16(&sQf[row][kD + col], sq8(R.q[s], 1.f));
                if constexpr (!DUAL) {
                    st16(&sKf[row][col], R.k[s]);
                    st16(&sKf[row][kD + col], sq8(R.k[s], 0.5f));
                    st16(&sV[row][col], R.v[s]);
                }
                st16(&sG[row][col], gr[s]);
                if (col == 0) {
                    sGd[row] = gdr[s];
                    sG[row][kD] = f32_to_bf16_bits(gdr[s]);
                }
            }
            if constexpr (!DUAL) {
#pragma unroll
                for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                    for (int nb = 0; nb < 5; ++nb) {
                        const int n = 16 * nb + c16;
                        if (n > kD) continue;
                        *reinterpret_cast<uint2 *>(&sW[n][16 * (2 * w + fi) + 4 * g]) =
                            uint2{pack2(st[fi][nb][0], st[fi][nb][1]), pack2(st[fi][nb][2], st[fi][nb][3])};
                    }
                if (g == 0) sW1[16 * w + c16] = w1;
            }
        };
        load_qkv<!DUAL>(R, a, b, h, c_end - 1, ra, col);
        prepare(c_end - 1);
        publish();
        if (c_end - 2 >= c_begin) load_qkv<!DUAL>(R, a, b, h, c_end - 2, ra, col);
        for (int c = c_end - 1; c >= c_begin; --c) {
            const int nvalid = min(kC, a.L - c * kC);
            __syncthreads();  // tiles of chunk c and W at its end in LDS
            // ---- W <- l^n W + (om phi_q)^T G with om_t = l^(t-c0+1) on the A operand's
            // token slots; W1 likewise from partial sums over all threads
            const float ln = sPw[nvalid];
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 5; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) st[fi][nb][r] *= ln;
            f32x4 dw1 = f32x4{0.f, 0.f, 0.f, 0.f};  // W1 increment of value block w: rows 0..2 = om parts
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                float om[8];
                {
                    const f32x4 o0 = *reinterpret_cast<const f32x4 *>(&sOm[32 * ks + 4 * g]);
                    const f32x4 o1 = *reinterpret_cast<const f32x4 *>(&sOm[32 * ks + 16 + 4 * g]);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        om[t] = o0[t];
                        om[4 + t] = o1[t];
                    }
                }
                // lane (g, c16): part min(c16, 3) of om at its eight token slots
                const int pr = min(c16, 3);
                const uint2 o0 = *reinterpret_cast<const uint2 *>(&sOmp[pr][32 * ks + 4 * g]);
                const uint2 o1 = *reinterpret_cast<const uint2 *>(&sOmp[pr][32 * ks + 16 + 4 * g]);
                const bf16x8 ompart = as_bf16x8(u32x4{o0.x, o0.y, o1.x, o1.y});
                bf16x8 aq[2];
#pragma unroll
                for (int fi = 0; fi < 2; ++fi) {
                    const uint16_t *p0 = &sQf[32 * ks + 4 * g + tr_r][16 * (2 * w + fi) + tr_c];
                    aq[fi] = scale_op(tr_op<false>(p0, p0 + 16 * kPT, 0).h, om);
                }
#pragma unroll
                for (int nb = 0; nb < 5; ++nb) {
                    const uint16_t *p0 = &sG[32 * ks + 4 * g + tr_r][16 * nb + tr_c];
                    const bf16x8 gb = tr_op<false>(p0, p0 + 16 * kPV, 0).h;
#pragma unroll
                    for (int fi = 0; fi < 2; ++fi) st[fi][nb] = mfma(aq[fi], gb, st[fi][nb]);
                    if (nb == w) dw1 = mfma(ompart, gb, dw1);  // wave-uniform
                }
            }
            {
                // W1[n] = sum_t om_t G_t[n]: value column 16w + c16 from the three om parts
                // (rows 0..2, lane group g = 0); the gden column (fp32) in every wave alike
                w1 = ln * w1 + ((dw1[0] + dw1[1]) + dw1[2]);
                w1g = ln * w1g + wave_sum(sPw[lane + 1] * sGd[lane]);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (c > c_begin) prepare(c - 1);
            __syncthreads();  // every read of chunk c's tiles and of W is done
            if (c > c_begin) {
                publish();
                __builtin_amdgcn_sched_barrier(0);
                if (c - 2 >= c_begin) load_qkv<!DUAL>(R, a, b, h, c - 2, ra, col);
            }
        }
        if constexpr (DUAL) {
            // the segment's contribution, in this kernel's convention
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 5; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int f = 16 * (2 * w + fi) + 4 * g + r, fr = f & (kD - 1), n = 16 * nb + c16;
                        if (n < kD) slot[(f < kD ? kWsS1 : kWsS2) + fr * kD + n] = st[fi][nb][r];
                        else if (n == kD) slot[(f < kD ? kWsK1 : kWsK2) + fr] = st[fi][nb][r];
                    }
            if (g == 0) slot[kWsS0 + 16 * w + c16] = w1;
            if (ut == 0) slot[kWsK0] = w1g;
            return;
        }
        // ---- the incoming state's adjoint: W after chunk 0 (S2, K2 rows halved back);
        // with segments the dual scan writes it
        if (a.ds1i && a.G == 1) {
#pragma unroll
            for (int fi = 0; fi < 2; ++fi)
#pragma unroll
                for (int nb = 0; nb < 5; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int f = 16 * (2 * w + fi) + 4 * g + r, fr = f & (kD - 1), n = 16 * nb + c16;
                        float x = st[fi][nb][r];
                        if (n == kD && a.dense_in) x += a.kcorr[static_cast<size_t>(seq) * kBwdCorr + f];
                        if (f >= kD) x *= 0.5f;
                        if (n < kD) (f < kD ? a.ds1i : a.ds2i)[so1 + fr * kD + n] = x;
                        else if (n == kD) (f < kD ? a.dk1i : a.dk2i)[so0 + fr] = x;
                    }
            if (g == 0) a.ds0i[so0 + 16 * w + c16] = w1;
            if (ut == 0) a.dk0i[seq] = w1g + (a.dense_in ? a.kcorr[static_cast<size_t>(seq) * kBwdCorr + kF] : 0.f);
        }
        return;
    }

    // ================ readout role: dk and dv of rows 16w..16w+15 of every chunk
    if constexpr (!DUAL) {
        const int jw = 16 * w + c16;  // this lane's key row of the transposed blocks
        float mask[4][4];  // l^(i-j) [i >= j] for i = 16ib + 4g + r, j = jw (sPw[n]: l^n rounded from fp64)
#pragma unroll
        for (int ib = 0; ib < 4; ++ib)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int d = 16 * ib + 4 * g + r - jw;
                mask[ib][r] = (ib >= w && d >= 0) ? sPw[max(d, 0)] : 0.f;
            }
        for (int c = c_end - 1; c >= c_begin; --c) {
            const int nvalid = min(kC, a.L - c * kC);
            __syncthreads();  // tiles of chunk c and W at its end in LDS
            // ---- A[i][jw] = mask (1 + phi_q(i) . phi_k(jw)) and P[i][jw] = mask (g_i . v_jw + gden_i), i blocks ib >= w
            f32x4 sc[4], pp[4];
#pragma unroll
            for (int ib = 0; ib < 4; ++ib) {
                sc[ib] = pp[ib] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (ib < w) continue;
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
                    sc[ib] = mfma(as_bf16x8(lds128(&sQf[16 * ib + c16][32 * ks + 8 * g])),
                                  as_bf16x8(lds128(&sKf[jw][32 * ks + 8 * g])), sc[ib]);
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
                    pp[ib] = mfma(as_bf16x8(lds128(&sG[16 * ib + c16][32 * ks + 8 * g])),
                                  as_bf16x8(lds128(&sV[jw][32 * ks + 8 * g])), pp[ib]);
                const f32x4 gd = *reinterpret_cast<const f32x4 *>(&sGd[16 * ib + 4 * g]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sc[ib][r] = mask[ib][r] * (1.0f + sc[ib][r]);
                    pp[ib][r] = mask[ib][r] * (pp[ib][r] + gd[r]);
                }
            }
            // tail weight l^(e-1-j) of row jw
            const float tjc = jw < nvalid ? sPw[nvalid - 1 - jw] : 0.f;
            const int64_t orow = b * a.g_sb + h * a.g_sh + static_cast<int64_t>(c * kC + opaque(jw)) * a.g_sl + 4 * g;
            // ---- dv of row jw, columns 16nb + 4g + r: A^T G + tail (phi_k W + W1)
            {
                f32x4 dvv[4];
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) dvv[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    if (2 * ks + 1 < w) continue;
                    const bf16x8 A = acc_op(sc[2 * ks], sc[2 * ks + 1]);
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb) {
                        const uint16_t *p0 = &sG[32 * ks + 4 * g + tr_r][16 * nb + tr_c];
                        dvv[nb] = mfma(tr_op<false>(p0, p0 + 16 * kPV, 0).h, A, dvv[nb]);
                    }
                }
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    float kf[8];
                    unpack8(lds128(&sKf[jw][32 * ks + 8 * g]), kf);
                    const bf16x8 A = as_bf16x8(pack8s(kf, tjc));
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb)
                        dvv[nb] = mfma(as_bf16x8(lds128(&sW[16 * nb + c16][32 * ks + 8 * g])), A, dvv[nb]);
                }
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) {
                    const f32x4 w1v = *reinterpret_cast<const f32x4 *>(&sW1[16 * nb + 4 * g]);
#pragma unroll
                    for (int r = 0; r < 4; ++r) dvv[nb][r] += tjc * w1v[r];
                }
                if (jw < nvalid) store_row16(a.dv, a.dt_g, a.g_vec, orow, dvv);
            }
            // ---- dphi_k of row jw, features 16fb + 4g + r: P^T phi_q + tail (W V')
            f32x4 dphi[8];
#pragma unroll
            for (int fb = 0; fb < 8; ++fb) dphi[fb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                if (2 * ks + 1 < w) continue;
                const bf16x8 A = acc_op(pp[2 * ks], pp[2 * ks + 1]);
#pragma unroll
                for (int fb = 0; fb < 8; ++fb) {
                    const uint16_t *p0 = &sQf[32 * ks + 4 * g + tr_r][16 * fb + tr_c];
                    dphi[fb] = mfma(tr_op<false>(p0, p0 + 16 * kPT, 0).h, A, dphi[fb]);
                }
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const bf16x8 A = perm_row_op(&sV[jw][0], ks, g, tjc);
#pragma unroll
                for (int fb = 0; fb < 8; ++fb) {
                    const uint16_t *p0 = &sW[32 * ks + 4 * g + tr_r][16 * fb + tr_c];
                    dphi[fb] = mfma(tr_op<false>(p0, p0 + 16 * kPT, 0).h, A, dphi[fb]);
                }
            }
            // ---- dk = dphi[k] + k dphi[k*k/2], the K column of W added to both
            if (jw < nvalid) {
                f32x4 dv[4];
#pragma unroll
                for (int fb = 0; fb < 4; ++fb) {
                    const f32x4 kv = unpack4(&sKf[jw][16 * fb + 4 * g]);
                    const f32x4 wa = unpack4(&sW[kD][16 * fb + 4 * g]), wb = unpack4(&sW[kD][kD + 16 * fb + 4 * g]);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        dv[fb][r] = (dphi[fb][r] + tjc * wa[r]) + kv[r] * (dphi[fb + 4][r] + tjc * wb[r]);
                }
                store_row16(a.dk, a.dt_g, a.g_vec, orow, dv);
            }
            __syncthreads();  // every read of chunk c's tiles and of W is done
        }
    }
}

// Reverse scan over segments, elementwise (one thread per (sequence, state
// element)): slot s holds segment s's contribution C_s on entry and the dual
// state at its end on exit: W_end(G-1) = dM_out, W_end(s-1) = l^len(s) W_end(s)
// + C_s; W_end(-1) is the incoming state's adjoint.
__global__ __launch_bounds__(256) void bwd_dual_scan_kernel(const BwdArgs a) {
    const int S = a.B * a.H;
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= static_cast<int64_t>(S) * kWsElems) return;
    const int seq = static_cast<int>(gid / kWsElems), e = static_cast<int>(gid % kWsElems);
    const int h = seq % a.H;
    // (selective: segment s's own log2 decay, beside its slot's state)
    const bool sel = a.logd != nullptr;
    const double ld = sel ? 1.0 : static_cast<double>(a.decay[h]);
    const float lT = sel ? 0.f : static_cast<float>(int_pow(ld, int64_t{kC} * a.cps));
    const float lLast = sel ? 0.f : static_cast<float>(int_pow(ld, a.L - (a.G - 1) * a.cps * kC));
    const float f2 = sel ? 1.0f : 2.0f;  // the kernels' factor on the second-order adjoints
    const size_t so1 = static_cast<size_t>(seq) * kD * kD, so0 = static_cast<size_t>(seq) * kD;
    // the element's place in the reference state, and the factor of this kernel's convention
    const float *src = nullptr;
    float *dst = nullptr;
    size_t off = 0;
    float fac = 1.0f;
    if (e < kWsS2) { src = a.ds1o; dst = a.ds1i; off = so1 + e; }
    else if (e < kWsS0) { src = a.ds2o; dst = a.ds2i; off = so1 + e - kWsS2; fac = f2; }
    else if (e < kWsK1) { src = a.ds0o; dst = a.ds0i; off = so0 + e - kWsS0; }
    else if (e < kWsK2) { src = a.dk1o; dst = a.dk1i; off = so0 + e - kWsK1; }
    else if (e < kWsK0) { src = a.dk2o; dst = a.dk2i; off = so0 + e - kWsK2; fac = f2; }
    else { src = a.dk0o; dst = a.dk0i; off = seq; }
    float carry = a.ds1o ? fac * src[off] : 0.f;
    float *slot = a.ws + static_cast<size_t>(seq) * a.G * kWsStride + e;
    for (int s = a.G - 1; s >= 0; --s) {
        const float cs = slot[static_cast<size_t>(s) * kWsStride];
        const float f = sel ? exp2f(slot[static_cast<size_t>(s) * kWsStride + kWsDecay - e]) : s == a.G - 1 ? lLast : lT;
        slot[static_cast<size_t>(s) * kWsStride] = carry;
        carry = f * carry + cs;
    }
    if (a.ds1i) dst[off] = carry / fac;
}

hipError_t launch_bwd_dual_scan(const BwdArgs &a, hipStream_t stream) {
    const int64_t n = static_cast<int64_t>(a.B) * a.H * kWsElems;
    const TimerEvents ts = timer_events(PRIME_KERNEL_BWD_DUAL_SCAN);
    hipExtLaunchKernelGGL(bwd_dual_scan_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, stream,
                          ts.start, ts.stop, 0, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) timer_drop(ts);
    return e;
}

void plan_backward_segments(int S, int L, int *G, int *cps, int per_cu) {
    const int NC = (L + kC - 1) / kC;
    int g = 1;
    const int cu = device_cus();
    if (per_cu == 2 && S > 0) {
        // bf16 passes, two workgroups per CU, in microseconds: a round of up to one
        // workgroup per CU costs 8 and 7.8 a chunk (both passes), of up to two 8 and 11;
        // segments add 16 for the scans and launches, 3 a chunk for the state-only and
        // dual passes (two units per CU before they slow each other) and 0.04 a slot.
        // Fitted to 15 shapes from 12 x 128 to 96 x 8192 with every count; the choice is
        // within 1 % of the best in each.  12 x 512: 8 segments 38 us, one 71; 12 x 1000:
        // 16 49, 2 107; 48 x 777: 7 70, one 111; 200 x 1024: one 138, 2 166.
        auto cost = [&](int u, int c) {
            const int64_t units = static_cast<int64_t>(S) * u, full = units / (2 * cu), rem = units % (2 * cu);
            double t = static_cast<double>(full) * (8.0 + 11.0 * c);
            if (rem) t += 8.0 + (rem <= cu ? 7.8 : 11.0) * c;
            if (u > 1)
                t += 16.0 + 3.0 * c * std::max(1.0, static_cast<double>(units) / (2.0 * cu)) +
                     0.04 * static_cast<double>(units);
            return t;
        };
        double best = cost(1, NC);
        for (int t = 2; t <= min(NC, 64); ++t) {
            const int c = (NC + t - 1) / t, u = (NC + c - 1) / c;
            if (cost(u, c) < best - 1e-9) {
                best = cost(u, c);
                g = u;
            }
        }
    } else if (S > 0) {
        // fp32 passes, one workgroup per CU: in periods of a chunk of the dq or dk/dv
        // pass (16-18 us each), a round of units over the CUs costs 2 a chunk, with
        // segments 2.6 (the state-only and dual passes) and about 1.2 for the two scans
        // and their slots' traffic.  96 sequences of 16 chunks: 8 segments 17.6 against 22
        // with 2; 48 sequences of 13: 5 segments 9.2 against 26 with one.
        double best = 1.9 * NC * ((S + cu - 1) / cu);  // (segments only where they pay by 5 %)
        g = 1;
        for (int t = 2; t <= min(NC, 64); ++t) {
            const int c = (NC + t - 1) / t, u = (NC + c - 1) / c;
            const double rounds = static_cast<double>((static_cast<int64_t>(S) * u + cu - 1) / cu);
            const double cost = 2.6 * rounds * c + 1.2 + 0.001 * S * u;
            if (cost < best - 1e-9) {
                best = cost;
                g = u;
            }
        }
    }
    if (g < 2) {
        *G = 1;
        *cps = NC;
        return;
    }
    const int c = (NC + g - 1) / g;
    *cps = c;
    *G = (NC + c - 1) / c;  // no empty segments
}

// gradient rows take one store of four elements if every row starts on such a boundary
bool gradient_rows_vec(const BwdArgs &a) {
    const uintptr_t four = (a.dt_g == PRIME_F32 ? 4 : 2) * 4;
    return (reinterpret_cast<uintptr_t>(a.dq) | reinterpret_cast<uintptr_t>(a.dk) | reinterpret_cast<uintptr_t>(a.dv)) %
                   four == 0 &&
           a.g_sb % 4 == 0 && a.g_sh % 4 == 0 && a.g_sl % 4 == 0;
}

hipError_t launch_prefill_backward(const BwdArgs &args, hipStream_t stream) {
    if (args.dt_in == PRIME_F32) return launch_prefill_backward_f32(args, stream);
    BwdArgs a = args;
    a.g_vec = gradient_rows_vec(a);
    const int S = a.B * a.H;
    hipError_t e;
    if (a.G > 1) {
        // the state entering every segment, by the forward's state-only pass and scan
        PrefillArgs f{};
        f.q = a.q; f.k = a.k; f.v = a.v;
        f.q_sb = a.q_sb; f.q_sh = a.q_sh; f.q_sl = a.q_sl;
        f.k_sb = a.k_sb; f.k_sh = a.k_sh; f.k_sl = a.k_sl;
        f.v_sb = a.v_sb; f.v_sh = a.v_sh; f.v_sl = a.v_sl;
        f.dt_in = a.dt_in; f.B = a.B; f.H = a.H; f.group = 1; f.L = a.L;
        f.decay = a.decay; f.eps = a.eps;
        f.s0i = a.s0i; f.s1i = a.s1i; f.s2i = a.s2i; f.k0i = a.k0i; f.k1i = a.k1i; f.k2i = a.k2i;
        f.G = a.G; f.cps = a.cps; f.ws = a.ws; f.states_only = 1;
        if ((e = launch_prefill(f, stream)) != hipSuccess) return e;
    }
    const int units = S * a.G;
    const TimerEvents t1 = timer_events(PRIME_KERNEL_BWD_DQ);
    if (a.dense_in)
        hipExtLaunchKernelGGL(prefill_bwd_dq_kernel<true>, dim3(units), dim3(512), 0, stream, t1.start, t1.stop, 0, a);
    else
        hipExtLaunchKernelGGL(prefill_bwd_dq_kernel<false>, dim3(units), dim3(512), 0, stream, t1.start, t1.stop, 0,
                              a);
    if ((e = hipGetLastError()) != hipSuccess) return timer_drop(t1), e;
    if (a.G > 1) {
        // each segment's dual contribution, then the reverse scan (slots now hold dual states)
        const TimerEvents td = timer_events(PRIME_KERNEL_BWD_DUAL);
        hipExtLaunchKernelGGL(prefill_bwd_dkv_kernel<true>, dim3(units), dim3(256), 0, stream, td.start, td.stop, 0,
                              a);
        if ((e = hipGetLastError()) != hipSuccess) return timer_drop(td), e;
        if ((e = launch_bwd_dual_scan(a, stream)) != hipSuccess) return e;
    }
    const TimerEvents t2 = timer_events(PRIME_KERNEL_BWD_DKV);
    hipExtLaunchKernelGGL(prefill_bwd_dkv_kernel<false>, dim3(units), dim3(512), 0, stream, t2.start, t2.stop, 0,
                          a);
    if ((e = hipGetLastError()) != hipSuccess) timer_drop(t2);
    return e;
}

}  // namespace prime
