// Chunked PRIME in fp32 throughout: the prefill of head dims below 64 and of
// selective PRIME with fp32 inputs (selective.py:363-365, 414-440), and the
// backward of both and of the base prefill with fp32 inputs -- the
// reverse-mode derivative of attention.py:119-143 (the recurrence the
// reference's prefill computes, chunked_ssd.py:48-184) that torch autograd
// takes when it trains in fp32 (tests/test_attention.py:50-62).
//
// Forward, per 64-token chunk with Fq_i = [q_i, q_i*q_i], Fk_j = [k_j, k_j*k_j/2]
// (k is beta k in the selective form), the state M = [S1; S2/2] (2D x D; [S1; S2] in
// the selective convention, whose S2 carries the 1/2), Kf likewise, and the decay
// from token j to token i written l(i, j), e_i that from the chunk's start through
// token i, w_j that from token j to the chunk's end (tokens past L: no weight, no
// decay):
//   a_ij  = [j <= i] l(i, j) (1 + Fq_i . Fk_j)
//   num_i = sum_j a_ij v_j + e_i (S0 + Fq_i M),  den_i = sum_j a_ij + e_i (K0 + Fq_i . Kf)
//   y_i   = num_i / D_i,  D_i = max(den_i, eps)
//   M <- e_63 M + Fk^T diag(w) V (likewise S0, K0, Kf)
// Backward, with g_i = dy_i / D_i and h_i = -[den_i >= eps] (dy_i . num_i) / D_i^2:
//   da_ij  = l(i, j) (g_i . v_j + h_i)                             (j <= i)
//   dFq_i  = sum_j da_ij Fk_j + e_i (M g_i + h_i Kf)                (state entering the chunk)
//   dv_j   = sum_i a_ij g_i + w_j (Fk_j dM + dS0)                  (adjoint dM, dS0, dKf of the
//   dFk_j  = sum_i da_ij Fq_i + w_j (dM v_j + dKf)                  state leaving the chunk)
//   dM    <- e_63 dM + Fq^T diag(e) G   (likewise dS0 from g, dK0 and dKf from h)
//   dq = dFq[:D] + 2 q * dFq[D:],  dk = dFk[:D] + k * dFk[D:]
// The base form's decays come from a table of powers of the head's decay (exact for
// any value, 0 included), the selective form's from the chunk's cumulative log decays.
//
// Three kernels (prefill, dq pass, dk/dv pass), one workgroup of 16 waves per
// (sequence, head) or segment of one, chunks in order (dk/dv: in reverse); every
// contraction is an fp32 MFMA (v_mfma_f32_16x16x4_f32: lane l holds A[l%16][l/16]
// and B[l/16][l%16], the accumulator D[4(l/16) + r][l%16]).  Head dims are padded
// with zeros to DP = 16, 32 or 64: zero columns of q, k and v add nothing to any sum.
// What bounds a chunk is its chain of phases, so the layout serves that:
// - 16 waves, one 16 x 16 unit of each phase per wave at DP = 64 (the pair of a
//   feature block and its squares is one unit, whose operands are read once: LDS
//   holds q and k, the squares are formed as they are read);
// - the next chunk's rows are loaded into registers a chunk ahead;
// - the denominators and the moments of a value that is always 1 (Kf, K0) and S0 are
//   VALU sums spread over all 1024 threads, beside the MFMA units;
// - the products with the carried state run beside the score tiles of their phase, the
//   products with a and da in the next;
// - LDS pitches by the way each array is read (Dim).
// Measured at D = 64, 96 sequences of 1000 tokens: dq pass 119 us, dk/dv 117, dual 47
// (8 waves, nothing loaded ahead, 2 segments: 187, 206, 72); a chunk is 16-18 us of which
// its MFMAs are 8.4.  At D = 32, 8 sequences of 256 tokens: prefill 25 us, backward 71 us, against
// 934 and 3580 us for one wavefront per sequence running the recurrence token by token
// (a single token, and a few tokens on many sequences, keep a kernel that goes token by token:
// generic_d.hip).

#include "f32_common.h"
#include "head_row.h"

namespace prime {
namespace {

constexpr int kT = 1024, kNW = kT / kWave;

template <int DP>
struct Dim {
    static constexpr int FP = 2 * DP;              // features
    static constexpr int ND = DP / 16;             // 16-wide blocks of a head row
    static constexpr int NE = kC * DP / kT;        // elements of a row array per thread
    // LDS pitches by how a wave reads the array (64 banks): 16 rows x 4 columns, 4
    // rows x 16 columns, or both ways (then 4 x 16 meets 12 banks twice)
    static constexpr int PR = DP == 64 ? 68 : DP == 32 ? 36 : 20;
    static constexpr int PC = DP == 64 ? 80 : DP == 32 ? 48 : 16;
    static constexpr int PB = DP == 64 ? 84 : DP == 32 ? 36 : 20;
};
constexpr int kPA = kC + 4, kPAt = kC + 16;  // a / da rows, read by rows (dq) or by columns (dk/dv)

// sum over the 16 lanes of a row of lanes, in each of them
__device__ __forceinline__ float sum16(float x) {
    x += xor_lane<1>(x);
    x += xor_lane<2>(x);
    x += xor_lane<4>(x);
    return x + xor_lane<8>(x);
}

// n batches of B k-steps: the next batch's LDS reads go out before this batch's
// MFMAs (left alone the compiler reads a whole unrolled loop's operands first and
// waits for them with the matrix cores idle).
template <int B, class T, class L, class M>
__device__ __forceinline__ void pipe(int n, L load, M mul) {
    T cur[B];
#pragma unroll
    for (int e = 0; e < B; ++e) cur[e] = load(e);
    for (int b = 1; b < n; ++b) {
        T nxt[B];
#pragma unroll
        for (int e = 0; e < B; ++e) nxt[e] = load(b * B + e);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < B; ++e) mul(cur[e]);
#pragma unroll
        for (int e = 0; e < B; ++e) cur[e] = nxt[e];
    }
#pragma unroll
    for (int e = 0; e < B; ++e) mul(cur[e]);
}
struct Op2 {
    float a, b;
};
struct Op3 {
    float a, b, c;
};
struct OpV {
    f32x4 a, b;
};

// NE consecutive elements of a row from column d0 as stored, from clamped addresses:
// nothing is masked or converted here, so that no wait sits between a load and the
// work it is to hide behind (a select on the loaded value cost half the dq pass).
template <int DP, bool VEC>
__device__ __forceinline__ void load_raw(const void *p, int dt, int64_t row, int d0, int D,
                                         uint32_t (&o)[Dim<DP>::NE]) {
    constexpr int NE = Dim<DP>::NE;
    if constexpr (VEC) {
        static_assert(NE == 4, "vector rows are 64 wide");
        const u32x4 x = *reinterpret_cast<const u32x4 *>(static_cast<const float *>(p) + row + d0);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[e];
    } else if (dt == PRIME_F32) {
#pragma unroll
        for (int e = 0; e < NE; ++e) o[e] = static_cast<const uint32_t *>(p)[row + min(d0 + e, D - 1)];
    } else {
#pragma unroll
        for (int e = 0; e < NE; ++e) o[e] = static_cast<const uint16_t *>(p)[row + min(d0 + e, D - 1)];
    }
}
// ... and as fp32, zero past D or when !valid
template <int DP, bool VEC>
__device__ __forceinline__ void to_f32(const uint32_t (&r)[Dim<DP>::NE], int dt, int d0, int D, bool valid,
                                       float (&o)[Dim<DP>::NE]) {
#pragma unroll
    for (int e = 0; e < Dim<DP>::NE; ++e) {
        float x = __uint_as_float(r[e]);
        if (dt == PRIME_BF16) x = __uint_as_float(r[e] << 16);
        else if (dt == PRIME_F16) x = h16_bits_to_f32(static_cast<uint16_t>(r[e]));
        o[e] = valid && (VEC || d0 + e < D) ? x : 0.f;
    }
}

template <int DP, int P>
__device__ __forceinline__ void put_elems(float (*s)[P], int i, int d0, const float (&x)[Dim<DP>::NE]) {
#pragma unroll
    for (int e = 0; e < Dim<DP>::NE; ++e) s[i][d0 + e] = x[e];
}

// NV = 1 or 4 consecutive values of an output row, masked past D
__device__ __forceinline__ void store_out(void *p, int dt, int64_t idx, f32x4 v, int nvalid, bool vec) {
    if (vec && dt == PRIME_F32) {
        st4(static_cast<float *>(p) + idx, v);
    } else if (vec && dt == PRIME_BF16) {
        *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(p) + idx) = uint2{pack2(v[0], v[1]), pack2(v[2], v[3])};
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r < nvalid) store_elem(p, idx + r, dt, v[r]);
    }
}

// A thread's share of a chunk's rows, loaded a chunk ahead
template <int DP>
struct Rows {
    uint32_t q[Dim<DP>::NE], k[Dim<DP>::NE], v[Dim<DP>::NE], dy[Dim<DP>::NE];
    float ld;  // wave 0, selective: the token's log decay
};

// (the chunk's first row is a scalar address and the row within it is formed from the
// chunk's length here: no per-thread 64-bit base is carried from chunk to chunk, whose
// spilled copies would be reloaded between the loads and wait for them)
template <int DP, bool VEC, bool SEL, bool DY, bool STATE_ONLY = false>
__device__ __forceinline__ void load_rows(const ChunkF32Args &a, int b, int h, int seq, int c, int tid, Rows<DP> &R) {
    const int d0 = Dim<DP>::NE * (tid & 15);
    const int last = min(kC, a.L - c * kC) - 1;
    const int64_t i = min(tid >> 4, last), t0 = static_cast<int64_t>(c) * kC;
    const int hk = h / a.group;
    auto row0 = [](const void *p, int dt, int64_t off) {
        return static_cast<const void *>(static_cast<const char *>(p) + off * (dt == PRIME_F32 ? 4 : 2));
    };
    if constexpr (!STATE_ONLY)
        load_raw<DP, VEC>(row0(a.q, a.dt_q, b * a.q_sb + h * a.q_sh + t0 * a.q_sl), a.dt_q, i * a.q_sl, d0, a.D, R.q);
    load_raw<DP, VEC>(row0(a.k, a.dt_k, b * a.k_sb + hk * a.k_sh + t0 * a.k_sl), a.dt_k, i * a.k_sl, d0, a.D, R.k);
    load_raw<DP, VEC>(row0(a.v, a.dt_v, b * a.v_sb + hk * a.v_sh + t0 * a.v_sl), a.dt_v, i * a.v_sl, d0, a.D, R.v);
    if constexpr (DY) {
        const void *p = row0(a.dy, a.dt_dy, b * a.dy_sb + h * a.dy_sh + t0 * a.dy_sl);
        if (VEC && a.dt_dy == PRIME_F32) load_raw<DP, VEC>(p, PRIME_F32, i * a.dy_sl, d0, a.D, R.dy);
        else load_raw<DP, false>(p, a.dt_dy, i * a.dy_sl, d0, a.D, R.dy);
    }
    if constexpr (SEL)
        if (tid < kWave) R.ld = (a.log_decay + static_cast<size_t>(seq) * a.L + t0)[min(tid, last)];
}
// A masked score is 0, and 0 times an infinity or NaN is NaN: the tile on the diagonal, whose
// product runs over 16 tokens, would carry such a value (or one whose square overflows) to
// tokens that do not see it.  The sum of squares of the operands of those products tells
// whether a chunk has one; it then takes the tiles token by token (diag_rows, diag_cols).
// At D = 64 with vector rows (VEC) it does not.
template <int DP>
__device__ __forceinline__ float add_squares(const float (&x)[Dim<DP>::NE], float s) {
#pragma unroll
    for (int e = 0; e < Dim<DP>::NE; ++e) s = fmaf(x[e], x[e], s);
    return s;
}

// the loaded rows in LDS as fp32 (k times kscale), zero past L and D; the sum of squares of
// those of q, k and v that SQ names (bits 0, 1, 2)
template <int DP, bool VEC, bool STATE_ONLY, int SQ, int PQ, int PK, int PV>
__device__ __forceinline__ float put_rows(const ChunkF32Args &a, const Rows<DP> &R, int i, int d0, int nv, float kscale,
                                          float (*sQ)[PQ], float (*sK)[PK], float (*sV)[PV]) {
    float x[Dim<DP>::NE], sq = 0.f;
    if constexpr (!STATE_ONLY) {
        to_f32<DP, VEC>(R.q, VEC ? PRIME_F32 : a.dt_q, d0, a.D, i < nv, x);
        put_elems<DP>(sQ, i, d0, x);
        if constexpr (!VEC && (SQ & 1)) sq = add_squares<DP>(x, sq);
    }
    to_f32<DP, VEC>(R.k, VEC ? PRIME_F32 : a.dt_k, d0, a.D, i < nv, x);
#pragma unroll
    for (int e = 0; e < Dim<DP>::NE; ++e) x[e] *= kscale;
    put_elems<DP>(sK, i, d0, x);
    if constexpr (!VEC && (SQ & 2)) sq = add_squares<DP>(x, sq);
    to_f32<DP, VEC>(R.v, VEC ? PRIME_F32 : a.dt_v, d0, a.D, i < nv, x);
    put_elems<DP>(sV, i, d0, x);
    if constexpr (!VEC && (SQ & 4)) sq = add_squares<DP>(x, sq);
    return sq;
}

// e^(a + b) for a in whole steps of kLogStep and |b| small: the rounding of the sum is put
// back as a factor
__device__ __forceinline__ float exp_sum(float a, float b) {
    const float d = a + b, e = expf(d), r = b - (d - a);
    return fabsf(r) < 1.f ? fmaf(e, r, e) : e;  // (not for infinities and NaN)
}

// The chunk's decays: sEc[i] = e_i, sW[j] = w_j (0 past L), and e_63, sum w in
// sSc[0], sSc[1]; selective: sCum, the cumulative log decays.  Wave 0.
//
// The selective decays are differences of prefix sums, and one strong decay makes every
// later sum large: in one fp32 number the mild decays after it keep the absolute error of
// that large sum (1.6e-5 of y with half the tokens at e^-25, against 1e-7 token by token).
// So each log decay is split at kLogStep = 2^-9: the sums of the steps are exact (at most 64 x
// 200 < 2^14, 23 bits), those of the rest stay below 2^-3.  sCum holds both, [0, 64) and
// [64, 128).
constexpr float kLogStep = 1.0f / 512;
template <bool SEL>
__device__ __forceinline__ void put_decays(int nv, int lane, float ld, const float *sPw, float *sCum, float *sEc,
                                           float *sW, float *sSc) {
    float e, w, e63;
    if constexpr (SEL) {
        // (e^-200 is 0 in fp32; -inf would make the differences NaN)
        const float x = lane < nv ? (ld < -200.f ? -200.f : ld) : 0.f;
        const float xs = rintf(x * (1.0f / kLogStep)) * kLogStep;
        const float cum = wave_prefix_sum(xs), low = wave_prefix_sum(x - xs);
        const float cend = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cum), 63));
        const float lend = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(low), 63));
        sCum[lane] = cum;
        sCum[kC + lane] = low;
        e = exp_sum(cum, low);
        w = lane < nv ? exp_sum(cend - cum, lend - low) : 0.f;
        e63 = exp_sum(cend, lend);
    } else {
        e = sPw[min(lane + 1, nv)];
        w = lane < nv ? sPw[nv - 1 - lane] : 0.f;
        e63 = sPw[nv];
    }
    sEc[lane] = e;
    sW[lane] = w;
    const float sw = wave_sum(w);
    if (lane == 0) {
        sSc[0] = e63;
        sSc[1] = sw;
    }
}

template <bool SEL>
__device__ __forceinline__ float decay_ij(int i, int j, const float *sPw, const float *sCum) {
    if constexpr (SEL) return exp_sum(sCum[i] - sCum[j], sCum[kC + i] - sCum[kC + j]);
    else return sPw[i - j];
}

// One lower tile of q . k and q^2 . k^2 / 2 over D (k-slot g of k-step s: D/4 g + s)
template <int DP, int PQ, int PK>
__device__ __forceinline__ f32x4 score_tile(int ib, int jb, int g, int c16, const float (*sQ)[PQ],
                                            const float (*sK)[PK]) {
    const float *pa = &sQ[16 * ib + c16][DP / 4 * g];
    const float *pb = &sK[16 * jb + c16][DP / 4 * g];
    f32x4 p = {0.f, 0.f, 0.f, 0.f}, p2 = {0.f, 0.f, 0.f, 0.f};
    pipe<1, OpV>(DP / 16, [&](int q4) { return OpV{ld4(pa + 4 * q4), ld4(pb + 4 * q4)}; },
                 [&](const OpV &o) {
#pragma unroll
                     for (int r = 0; r < 4; ++r) {
                         p = mfma4(o.a[r], o.b[r], p);
                         p2 = mfma4(o.a[r] * o.a[r], 0.5f * (o.b[r] * o.b[r]), p2);
                     }
                 });
    return p + p2;
}

// a on lower tile w, masked to valid columns
template <int DP, bool SEL, int PQ, int PK, int PA>
__device__ __forceinline__ void put_scores(int w, int nv, int g, int c16, const float (*sQ)[PQ], const float (*sK)[PK],
                                           const float *sPw, const float *sCum, float (*sA)[PA]) {
    int ib, jb;
    lower_tile(w, ib, jb);
    const f32x4 p = score_tile<DP, PQ, PK>(ib, jb, g, c16, sQ, sK);
    const int j = 16 * jb + c16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 16 * ib + 4 * g + r;
        sA[i][j] = (i >= j && j < nv) ? decay_ij<SEL>(i, j, sPw, sCum) * (1.0f + p[r]) : 0.f;
    }
}

// da on lower tile w: l(i, j) (g_i . v_j + h_i), masked like a
template <int DP, bool SEL, int PG, int PV>
__device__ __forceinline__ f32x4 dscore_tile(int w, int nv, int g, int c16, const float (*sG)[PG],
                                             const float (*sV)[PV], const float *sH, const float *sPw,
                                             const float *sCum) {
    int ib, jb;
    lower_tile(w, ib, jb);
    f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q4 = 0; q4 < DP / 16; ++q4) {
        const f32x4 x = ld4(&sG[16 * ib + c16][DP / 4 * g + 4 * q4]), z = ld4(&sV[16 * jb + c16][DP / 4 * g + 4 * q4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) p = mfma4(x[r], z[r], p);
    }
    const int j = 16 * jb + c16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 16 * ib + 4 * g + r;
        p[r] = (i >= j && j < nv) ? decay_ij<SEL>(i, j, sPw, sCum) * (p[r] + sH[i]) : 0.f;
    }
    return p;
}
template <int PA>
__device__ __forceinline__ void put_tile(int w, int g, int c16, f32x4 p, float (*sA)[PA]) {
    int ib, jb;
    lower_tile(w, ib, jb);
#pragma unroll
    for (int r = 0; r < 4; ++r) sA[16 * ib + 4 * g + r][16 * jb + c16] = p[r];
}

// the powers of the head's decay, l^0 .. l^64 (rounded once)
__device__ __forceinline__ void put_powers(const ChunkF32Args &a, int h, int tid, float *sPw) {
    if (tid <= kC) sPw[tid] = static_cast<float>(pow_sum(a.decay[h], tid).p);
}

// A state in the layout of the kernels: unit (db, dv) of M's two halves in a
// wave's accumulators, Kf[f] in threads f = tid / (kT / 128) .., S0 likewise.
struct StatePtrs {
    const float *s0, *s1, *s2, *k0, *k1, *k2;
};
// the state of sequence seq, or of a segment's slot (D = 64)
__device__ __forceinline__ StatePtrs seq_state(const float *s0, const float *s1, const float *s2, const float *k0,
                                               const float *k1, const float *k2, int seq, int D) {
    if (!s1) return StatePtrs{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    const size_t o1 = static_cast<size_t>(seq) * D * D, o0 = static_cast<size_t>(seq) * D;
    return StatePtrs{s0 + o0, s1 + o1, s2 + o1, k0 + seq, k1 + o0, k2 + o0};
}
__device__ __forceinline__ StatePtrs slot_state(const float *slot) {
    return StatePtrs{slot + kWsS0, slot + kWsS1, slot + kWsS2, slot + kWsK0, slot + kWsK1, slot + kWsK2};
}

// The carried moments of one workgroup: this wave's unit of M (two halves) and
// this thread's Kf, S0 and K0 elements.
template <int DP>
struct Carry {
    f32x4 m[2];
    float kf, s0, k0;
};
template <int DP>
__device__ __forceinline__ bool has_unit(int u) { return u < Dim<DP>::ND * Dim<DP>::ND; }

// c2: the factor between the state's second-order components and M's rows D ..
template <int DP>
__device__ __forceinline__ void load_carry(const StatePtrs &p, int D, float c2, int u, int g, int c16, int tid,
                                           Carry<DP> &C) {
    constexpr int ND = Dim<DP>::ND;
    C.kf = C.s0 = C.k0 = 0.f;
    C.m[0] = C.m[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!p.s1) return;
    if (has_unit<DP>(u)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int f = 16 * (u / ND) + 4 * g + r, col = 16 * (u % ND) + c16;
            if (f < D && col < D) {
                C.m[0][r] = p.s1[f * D + col];
                C.m[1][r] = c2 * p.s2[f * D + col];
            }
        }
    }
    const int f = tid >> 3, d = tid >> 4;
    if (f < 2 * DP && (f & (DP - 1)) < D) C.kf = f < DP ? p.k1[f] : c2 * p.k2[f - DP];
    if (d < DP && d < D) C.s0 = p.s0[d];
    C.k0 = p.k0[0];
}
template <int DP, int PM>
__device__ __forceinline__ void publish(const Carry<DP> &C, int u, int g, int c16, int tid, float (*sM)[PM], float *sKf,
                                        float *sS0) {
    constexpr int ND = Dim<DP>::ND;
    if (has_unit<DP>(u)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            sM[16 * (u / ND) + 4 * g + r][16 * (u % ND) + c16] = C.m[0][r];
            sM[DP + 16 * (u / ND) + 4 * g + r][16 * (u % ND) + c16] = C.m[1][r];
        }
    }
    if ((tid & 7) == 0 && (tid >> 3) < 2 * DP) sKf[tid >> 3] = C.kf;
    if ((tid & 15) == 0 && (tid >> 4) < DP) sS0[tid >> 4] = C.s0;
}
// (the pointers of p are written here)
template <int DP>
__device__ __forceinline__ void store_carry(const StatePtrs &p, int D, float c2, int u, int g, int c16, int tid,
                                            const Carry<DP> &C) {
    constexpr int ND = Dim<DP>::ND;
    auto w = [](const float *x) { return const_cast<float *>(x); };
    if (has_unit<DP>(u)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int f = 16 * (u / ND) + 4 * g + r, col = 16 * (u % ND) + c16;
            if (f < D && col < D) {
                w(p.s1)[f * D + col] = C.m[0][r];
                w(p.s2)[f * D + col] = c2 * C.m[1][r];
            }
        }
    }
    const int f = tid >> 3, d = tid >> 4;
    if ((tid & 7) == 0 && f < 2 * DP && (f & (DP - 1)) < D) {
        if (f < DP) w(p.k1)[f] = C.kf;
        else w(p.k2)[f - DP] = c2 * C.kf;
    }
    if ((tid & 15) == 0 && d < DP && d < D) w(p.s0)[d] = C.s0;
    if (tid == 0) w(p.k0)[0] = C.k0;
}

// C <- e63 C + F^T diag(x) V over the chunk: F = [r, c2 r*r] of the rows sR, the value
// rows sX weighted by sWt; Kf from sWk (the weight of the constant value), S0, K0.
// SECOND: the factor on the squares.
template <int DP, int PR, int PX>
__device__ __forceinline__ void advance(Carry<DP> &C, float second, float e63, float sumk, int u, int g, int c16,
                                        int tid, const float (*sR)[PR], const float (*sX)[PX], const float *sWt,
                                        const float *sWk) {
    constexpr int ND = Dim<DP>::ND;
    if (has_unit<DP>(u)) {
        f32x4 x = C.m[0] * e63, y = C.m[1] * e63;
        const int fc = 16 * (u / ND) + c16, xc = 16 * (u % ND) + c16;
        pipe<4, Op3>(
            4, [&](int s) { return Op3{sR[4 * s + g][fc], sWt[4 * s + g], sX[4 * s + g][xc]}; },
            [&](const Op3 &o) {
                const float vv = o.b * o.c;
                x = mfma4(o.a, vv, x);
                y = mfma4(second * (o.a * o.a), vv, y);
            });
        C.m[0] = x;
        C.m[1] = y;
    }
    // 8 threads a feature, 16 a value column
    if (tid < 16 * DP) {
        const int f = tid >> 3, part = tid & 7;
        float t = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int j = part + 8 * e;
            const float x = sR[j][f & (DP - 1)];
            t = fmaf(sWk[j], f < DP ? x : second * (x * x), t);
        }
        t += xor_lane<1>(t);
        t += xor_lane<2>(t);
        t += xor_lane<4>(t);
        C.kf = e63 * C.kf + t;
        const int d = tid >> 4, p16 = tid & 15;
        t = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = p16 + 16 * e;
            t = fmaf(sWt[j], sX[j][d], t);
        }
        C.s0 = e63 * C.s0 + sum16(t);
    }
    C.k0 = e63 * C.k0 + sumk;
}

// this thread's 16th of token i's Fq . Kf
template <int DP, int PQ>
__device__ __forceinline__ float k_readout(int i, int part, const float (*sQ)[PQ], const float *sKf) {
    constexpr int NE = Dim<DP>::NE;
    float rd = 0.f;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        const float q = sQ[i][NE * part + e];
        rd = fmaf(q, sKf[NE * part + e], rd);
        rd = fmaf(q * q, sKf[DP + NE * part + e], rd);
    }
    return rd;
}

// The diagonal tile of block tb token by token: x[r] += sum over j <= tok of a[tok][j] times
// the row's column 16 xb + 4 g + r ...
template <int PX, int PA>
__device__ __forceinline__ void diag_rows(int tb, int xb, int g, int tok, const float (*sX)[PX], const float (*sA)[PA],
                                          f32x4 &x) {
    for (int j = 16 * tb; j <= tok; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = fmaf(sA[tok][j], sX[j][16 * xb + 4 * g + r], x[r]);
}
// ... or over i >= tok of a[i][tok]
template <int PX, int PA>
__device__ __forceinline__ void diag_cols(int tb, int xb, int g, int tok, const float (*sX)[PX], const float (*sA)[PA],
                                          f32x4 &x) {
    for (int i = tok; i < 16 * tb + 16; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = fmaf(sA[i][tok], sX[i][16 * xb + 4 * g + r], x[r]);
}

// num^T tile of (token block tb, value block dv): the state's part (needs no scores) ...
template <int DP, int PQ, int PM>
__device__ __forceinline__ f32x4 num_state(int tb, int dv, int g, int c16, float ec, const float (*sQ)[PQ],
                                           const float (*sM)[PM], const float *sS0) {
    const int tok = 16 * tb + c16;
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
    pipe<4, Op3>(
        DP / 16,
        [&](int s) { return Op3{sQ[tok][4 * s + g], sM[4 * s + g][16 * dv + c16], sM[DP + 4 * s + g][16 * dv + c16]}; },
        [&](const Op3 &o) {
            const float eq = ec * o.a;
            x = mfma4(o.b, eq, x);
            y = mfma4(o.c, eq * o.a, y);
        });
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] += y[r] + ec * sS0[16 * dv + 4 * g + r];
    return x;
}
// ... and the chunk's values (a is zero above token 16 tb + 15)
template <int PV, int PA>
__device__ __forceinline__ f32x4 num_values(int tb, int dv, int g, int c16, const float (*sV)[PV],
                                            const float (*sA)[PA], f32x4 x, bool bad) {
    const int tok = 16 * tb + c16;
    const int n = bad ? tb : tb + 1;
    if (n)
        pipe<4, Op2>(n, [&](int s) { return Op2{sV[4 * s + g][16 * dv + c16], sA[tok][4 * s + g]}; },
                     [&](const Op2 &o) { x = mfma4(o.a, o.b, x); });
    if (bad) diag_rows(tb, dv, g, tok, sV, sA, x);
    return x;
}

}  // namespace

// ---------------------------------------------------------------------------
// Prefill.  DIN: the dense branch's double clamp with an incoming state (the
// call's own K moments are carried from zero, the incoming ones kept apart);
// VEC: D = 64 fp32 rows on 16-byte boundaries; STATE_ONLY (D = 64): a segment's
// state from zero (selective: and its log decay) into its slot.
// ---------------------------------------------------------------------------
template <int DP, bool DIN, bool SEL, bool VEC, bool STATE_ONLY>
__global__ __launch_bounds__(kT, 1) void chunk_f32_prefill_kernel(const ChunkF32Args a) {
    using K = Dim<DP>;
    __shared__ __attribute__((aligned(16))) float sQ[STATE_ONLY ? 1 : kC][K::PR];
    __shared__ __attribute__((aligned(16))) float sK[kC][K::PC];
    __shared__ __attribute__((aligned(16))) float sV[kC][K::PC];
    __shared__ __attribute__((aligned(16))) float sA[STATE_ONLY ? 1 : kC][kPA];
    __shared__ __attribute__((aligned(16))) float sM[STATE_ONLY ? 1 : K::FP][K::PB];
    __shared__ float sKf[K::FP], sKin[K::FP], sS0[DP], sPw[kC + 1], sCum[2 * kC], sEc[kC], sW[kC], sDen[kC], sSc[2];
    __shared__ int sBad;  // (!VEC) 1 + the last chunk with an infinite or NaN operand

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, c16 = lane & 15;
    const int nseg = STATE_ONLY ? a.G - 1 : a.G;  // the state-only pass takes segments 0 .. G-2
    const int unit = blockIdx.x;
    const int seq = unit / nseg, seg = unit - seq * nseg;
    const int b = seq / a.H, h = seq - b * a.H;
    const int u = kNW - 1 - w;  // this wave's unit of M (the scores take the low waves)
    float *slot = a.G > 1 ? a.slots + (static_cast<size_t>(seq) * a.G + seg) * kWsStride : nullptr;
    const float c2in = SEL ? 1.0f : 0.5f, c2out = SEL ? 1.0f : 2.0f;

    StatePtrs in = seq_state(a.s0i, a.s1i, a.s2i, a.k0i, a.k1i, a.k2i, seq, a.D);
    if (slot) in = slot_state(slot);
    if (STATE_ONLY) in.s1 = nullptr;
    Carry<DP> C;
    load_carry<DP>(in, a.D, c2in, u, g, c16, tid, C);
    float k0in = 0.f, kfin = 0.f;
    if constexpr (DIN) {
        kfin = C.kf;
        k0in = C.k0;
        if ((tid & 7) == 0 && (tid >> 3) < K::FP) sKin[tid >> 3] = kfin;
        C.kf = C.k0 = 0.f;
    }
    if constexpr (!SEL) put_powers(a, h, tid, sPw);

    const int NC = (a.L + kC - 1) / kC;
    const int c_begin = seg * a.cps, c_end = min(c_begin + a.cps, NC);
    const int i = tid >> 4, part = tid & 15, d0 = K::NE * part;
    float seg_ld = 0.f;
    double l64 = 1.0, lcd = 1.0;  // (DIN) l^64, l^(64 c)
    if constexpr (DIN) l64 = int_pow(a.decay[h], kC);
    Rows<DP> R;
    load_rows<DP, VEC, SEL, false, STATE_ONLY>(a, b, h, seq, c_begin, tid, R);
    if constexpr (!VEC) {
        if (tid == 0) sBad = 0;
    }
    if constexpr (!SEL || !VEC) __syncthreads();  // sPw, sBad
    for (int c = c_begin; c < c_end; ++c) {
        const int nv = min(kC, a.L - c * kC);
        if constexpr (!STATE_ONLY) publish<DP>(C, u, g, c16, tid, sM, sKf, sS0);
        const float sq =
            put_rows<DP, VEC, STATE_ONLY, 4>(a, R, i, d0, nv, SEL && !a.qk_norm ? a.k_scale[h] : 1.0f, sQ, sK, sV);
        if (!VEC && !(sq < INFINITY)) sBad = c + 1;
        if (w == 0) {
            put_decays<SEL>(nv, lane, R.ld, sPw, sCum, sEc, sW, sSc);
            if (SEL && STATE_ONLY) seg_ld += wave_sum(lane < nv ? R.ld : 0.f);
        }
        __syncthreads();
        if constexpr (!VEC && !STATE_ONLY) {
            if (a.qk_norm) {  // a row per thread, the order of prime_head_layernorm
                if (tid < nv) {
                    generic_ln_row(sQ[tid], a.D, a.qn_w, a.qn_b, a.dt_norm, a.ln_eps, a.q_scale, a.dt_q);
                } else if (tid >= kC && tid < kC + nv) {
                    float *row = sK[tid - kC];
                    generic_ln_row(row, a.D, a.kn_w, a.kn_b, a.dt_norm, a.ln_eps, 1.0f, a.dt_k);
                    if constexpr (SEL)
                        for (int d = 0; d < a.D; ++d) row[d] *= a.k_scale[h];
                }
                __syncthreads();
            }
        }
        if (c + 1 < c_end) load_rows<DP, VEC, SEL, false, STATE_ONLY>(a, b, h, seq, c + 1, tid, R);
        const float e63 = sSc[0], sumw = sSc[1];
        if constexpr (!STATE_ONLY) {
            const int tb = w / K::ND, dv = w % K::ND, tok = 16 * tb + c16;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            if (w < 4 * K::ND) acc = num_state<DP>(tb, dv, g, c16, sEc[tok], sQ, sM, sS0);
            if (w < 10) put_scores<DP, SEL>(w, nv, g, c16, sQ, sK, sPw, sCum, sA);
            __syncthreads();
            // ---- denominators, 16 threads a token (only a's lower tiles exist)
            {
                float p = 0.f;
                if ((part >> 2) <= (i >> 4)) {
                    const f32x4 x = ld4(&sA[i][4 * part]);
                    p = (x[0] + x[1]) + (x[2] + x[3]);
                }
                const float rd = k_readout<DP>(i, part, sQ, sKf);
                p = sum16(p + sEc[i] * rd) + sEc[i] * C.k0;
                float den = fmaxf(p, a.eps);
                if constexpr (DIN) {
                    // max(max(den of the call, eps) + l^(t+1) den_in, eps)
                    const float lc = static_cast<float>(lcd);
                    lcd *= l64;
                    const float ri = sum16(k_readout<DP>(i, part, sQ, sKin)) + k0in;
                    den = fmaxf(den + lc * sEc[i] * ri, a.eps);
                }
                if (part == 0) sDen[i] = den;
            }
            if (w < 4 * K::ND) acc = num_values(tb, dv, g, c16, sV, sA, acc, !VEC && __builtin_amdgcn_readfirstlane(sBad) == c + 1);
            advance<DP>(C, 0.5f, e63, sumw, u, g, c16, tid, sK, sV, sW, sW);
            __syncthreads();
            if (w < 4 * K::ND && tok < nv) {
                const float den = sDen[tok];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] = acc[r] / den;
                const int d = 16 * dv + 4 * g;
                store_out(a.y, a.dt_y, b * a.y_sb + h * a.y_sh + static_cast<int64_t>(c * kC + tok) * a.y_sl + d, acc,
                          a.D - d, VEC);
            }
        } else {
            advance<DP>(C, 0.5f, e63, sumw, u, g, c16, tid, sK, sV, sW, sW);
            __syncthreads();
        }
    }
    if constexpr (STATE_ONLY) {
        store_carry<DP>(slot_state(slot), a.D, c2out, u, g, c16, tid, C);
        if (SEL && tid == 0) slot[kWsDecay] = seg_ld * 1.44269504088896341f;  // log2
        return;
    }
    if (a.s1o && seg == a.G - 1) {
        if constexpr (DIN) {
            const float lL = static_cast<float>(int_pow(a.decay[h], a.L));
            C.kf += lL * kfin;
            C.k0 += lL * k0in;
        }
        store_carry<DP>(seq_state(a.s0o, a.s1o, a.s2o, a.k0o, a.k1o, a.k2o, seq, a.D), a.D, c2out, u, g, c16, tid, C);
    }
}

// ---------------------------------------------------------------------------
// dq pass: chunks in order, the forward state carried; leaves 1/D and h per
// token.  DIN: the dense double clamp with an incoming state; it also leaves the
// share of the incoming K adjoint that the inner clamp withholds from the call's
// tokens (kc1, kc2, kc0), which the dk/dv pass adds to that adjoint.  SEL:
// also per token phi_q'(i) . dphi_q'(i) (the query side of the log decays' adjoint,
// phi_q' = [1, q, q*q]) and per sequence <dstate_out, state_out>.
// ---------------------------------------------------------------------------
template <int DP, bool DIN, bool SEL, bool VEC>
__global__ __launch_bounds__(kT, 1) void chunk_f32_dq_kernel(const ChunkF32Args a) {
    using K = Dim<DP>;
    __shared__ __attribute__((aligned(16))) float sQ[kC][K::PR];
    __shared__ __attribute__((aligned(16))) float sK[kC][K::PC];
    __shared__ __attribute__((aligned(16))) float sV[kC][K::PC];
    __shared__ __attribute__((aligned(16))) float sG[kC][K::PR];  // dy, then g
    __shared__ __attribute__((aligned(16))) float sA[kC][kPA];    // a, then da
    __shared__ __attribute__((aligned(16))) float sM[K::FP][K::PB];
    __shared__ float sKf[K::FP], sS0[DP], sPw[kC + 1], sCum[2 * kC], sEc[kC], sW[kC], sH[kC], sSc[2];
    __shared__ float sPart[K::ND][kC];
    // dense double clamp: the incoming Kf, l^(64c) times the outer clamp's adjoint, and
    // l^(t+1) times the part of it the inner clamp withholds from the call's tokens
    __shared__ float sKin[K::FP], sHc[kC], sDh[kC];
    __shared__ float sFin[kNW];
    __shared__ int sBad;  // (!VEC) 1 + the last chunk with an infinite or NaN operand

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, c16 = lane & 15;
    const int unit = blockIdx.x;
    const int seq = unit / a.G, seg = unit - seq * a.G;
    const int b = seq / a.H, h = seq - b * a.H;
    const int u = kNW - 1 - w;
    const float c2in = SEL ? 1.0f : 0.5f;

    StatePtrs in = seq_state(a.s0i, a.s1i, a.s2i, a.k0i, a.k1i, a.k2i, seq, a.D);
    if (a.G > 1) in = slot_state(a.slots + static_cast<size_t>(unit) * kWsStride);
    Carry<DP> C;
    load_carry<DP>(in, a.D, c2in, u, g, c16, tid, C);
    float k0in = 0.f, corr = 0.f, corr0 = 0.f;
    double l64 = 1.0, lcd = 1.0;  // l^64, l^(64 c)
    if constexpr (DIN) {
        if ((tid & 7) == 0 && (tid >> 3) < K::FP) sKin[tid >> 3] = C.kf;
        k0in = C.k0;
        C.kf = C.k0 = 0.f;
        l64 = int_pow(a.decay[h], kC);
    }
    if constexpr (!SEL) put_powers(a, h, tid, sPw);

    const int NC = (a.L + kC - 1) / kC;
    const int c_begin = seg * a.cps, c_end = min(c_begin + a.cps, NC);
    const int i = tid >> 4, part = tid & 15, d0 = K::NE * part;
    const int64_t gbase = b * a.g_sb + h * a.g_sh;
    const int tb = w / K::ND, xb = w % K::ND, tok = 16 * tb + c16;  // this wave's unit of num and dFq
    Rows<DP> R;
    load_rows<DP, VEC, SEL, true>(a, b, h, seq, c_begin, tid, R);
    if constexpr (!VEC) {
        if (tid == 0) sBad = 0;
    }
    if constexpr (!SEL || !VEC) __syncthreads();
    for (int c = c_begin; c < c_end; ++c) {
        const int nv = min(kC, a.L - c * kC);
        {
            float x[K::NE];
            to_f32<DP, VEC>(R.dy, a.dt_dy, d0, a.D, i < nv, x);
            put_elems<DP>(sG, i, d0, x);
        }
        const float sq = put_rows<DP, VEC, false, 6>(a, R, i, d0, nv, SEL ? a.k_scale[h] : 1.0f, sQ, sK, sV);
        if (!VEC && !(sq < INFINITY)) sBad = c + 1;
        publish<DP>(C, u, g, c16, tid, sM, sKf, sS0);
        if (w == 0) put_decays<SEL>(nv, lane, R.ld, sPw, sCum, sEc, sW, sSc);
        __syncthreads();
        if (c + 1 < c_end) load_rows<DP, VEC, SEL, true>(a, b, h, seq, c + 1, tid, R);
        f32x4 num = {0.f, 0.f, 0.f, 0.f};
        if (w < 4 * K::ND) num = num_state<DP>(tb, xb, g, c16, sEc[tok], sQ, sM, sS0);
        if (w < 10) put_scores<DP, SEL>(w, nv, g, c16, sQ, sK, sPw, sCum, sA);
        __syncthreads();
        // ---- denominators (16 threads a token, all holding the result) and the dot num . dy
        const float ei = sEc[i];
        float den, d1;  // the call's denominator; plus the incoming term, each as clamped before
        float lc = 0.f;
        {
            float p = 0.f;
            if ((part >> 2) <= (i >> 4)) {
                const f32x4 x = ld4(&sA[i][4 * part]);
                p = (x[0] + x[1]) + (x[2] + x[3]);
            }
            const float rd = k_readout<DP>(i, part, sQ, sKf);
            den = sum16(p + ei * rd) + ei * C.k0;
            d1 = den;
            if constexpr (DIN) {
                lc = static_cast<float>(lcd);
                lcd *= l64;
                const float ri = sum16(k_readout<DP>(i, part, sQ, sKin)) + k0in;
                d1 = fmaxf(den, a.eps) + lc * ei * ri;
            }
        }
        if (w < 4 * K::ND) {
            num = num_values(tb, xb, g, c16, sV, sA, num, !VEC && __builtin_amdgcn_readfirstlane(sBad) == c + 1);
            const f32x4 dy = ld4(&sG[tok][16 * xb + 4 * g]);
            float dot = (dy[0] * num[0] + dy[1] * num[1]) + (dy[2] * num[2] + dy[3] * num[3]);
            dot = sum_lane32(sum_lane16(dot));
            if (g == 0) sPart[xb][tok] = dot;
        }
        __syncthreads();
        // ---- g = dy / D, h = -[den >= eps] (dy . num) / D^2; 1/D and h to the workspace
        {
            float dot = 0.f;
#pragma unroll
            for (int n = 0; n < K::ND; ++n) dot += sPart[n][i];
            const float D = fmaxf(d1, a.eps);
            const bool valid = i < nv;
            const float hout = valid && d1 >= a.eps ? -dot / (D * D) : 0.f;  // the outer clamp's adjoint
            const float hh = den >= a.eps ? hout : 0.f;                      // the call's share (inner clamp)
#pragma unroll
            for (int e = 0; e < K::NE; ++e) sG[i][d0 + e] = valid ? sG[i][d0 + e] / D : 0.f;
            if (part == 0) {
                sH[i] = hh;
                if constexpr (DIN) {
                    sHc[i] = lc * hout;
                    sDh[i] = lc * ei * (hout - hh);
                }
                if (valid) {
                    const size_t o = static_cast<size_t>(seq) * a.L + c * kC + i;
                    a.inv_den[o] = 1.0f / D;
                    a.g_den[o] = hh;
                    // SEL: phi_q'(i) . dphi_q'(i) = (num . dy) / D + den h.  e_i scales num and den alike,
                    // so this is exactly 0 while den >= eps (h = -(num . dy) / den^2) and (num . dy) /
                    // eps where the clamp holds (h = 0): without the cancellation of a sum over features
                    if constexpr (SEL) a.pq[o] = den >= a.eps ? 0.f : dot / D;
                }
            }
        }
        __syncthreads();
        const float e63 = sSc[0], sumw = sSc[1];
        // ---- dFq (token block tb; feature block xb and its squares): the state's part
        const float ec = sEc[tok];
        f32x4 fx = {0.f, 0.f, 0.f, 0.f}, fy = {0.f, 0.f, 0.f, 0.f};
        if (w < 4 * K::ND) {
            pipe<4, Op3>(
                DP / 16,
                [&](int s) {
                    return Op3{sG[tok][4 * s + g], sM[16 * xb + c16][4 * s + g], sM[DP + 16 * xb + c16][4 * s + g]};
                },
                [&](const Op3 &o) {
                    const float eg = ec * o.a;
                    fx = mfma4(o.b, eg, fx);
                    fy = mfma4(o.c, eg, fy);
                });
        }
        if (w < 10) {
            const f32x4 p = dscore_tile<DP, SEL>(w, nv, g, c16, sG, sV, sH, sPw, sCum);
            put_tile(w, g, c16, p, sA);
        }
        // (the vectors and M in LDS keep the state entering the chunk until the next publish)
        advance<DP>(C, 0.5f, e63, sumw, u, g, c16, tid, sK, sV, sW, sW);
        if constexpr (DIN) {  // sum over the chunk of sDh_t [Fq(t) | 1]
            if (tid < 16 * DP) {
                const int f = tid >> 3, p8 = tid & 7;
#pragma unroll 2
                for (int e = 0; e < 8; ++e) {
                    const float x = sQ[p8 + 8 * e][f & (DP - 1)];
                    corr = fmaf(sDh[p8 + 8 * e], f < DP ? x : x * x, corr);
                }
            }
            corr0 += wave_sum(sDh[lane]);
        }
        __syncthreads();
        // ---- dFq: the chunk's part -> dq
        if (w < 4 * K::ND) {
            const bool bad = !VEC && __builtin_amdgcn_readfirstlane(sBad) == c + 1;
            const int n = bad ? tb : tb + 1;
            if (n)
                pipe<4, Op2>(n, [&](int s) { return Op2{sK[4 * s + g][16 * xb + c16], sA[tok][4 * s + g]}; },
                             [&](const Op2 &o) {
                                 fx = mfma4(o.a, o.b, fx);
                                 fy = mfma4(0.5f * (o.a * o.a), o.b, fy);
                             });
            if (bad) {
                diag_rows(tb, xb, g, tok, sK, sA, fx);
                for (int j = 16 * tb; j <= tok; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float k = sK[j][16 * xb + 4 * g + r];
                        fy[r] = fmaf(0.5f * (k * k), sA[tok][j], fy[r]);
                    }
            }
            if (tok < nv) {
                const int d = 16 * xb + 4 * g;
                const f32x4 q = ld4(&sQ[tok][d]);
                const float hh = ec * sH[tok];
                f32x4 dq;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float x1 = fx[r] + hh * sKf[d + r], y1 = fy[r] + hh * sKf[DP + d + r];
                    if constexpr (DIN) {  // the incoming K's denominator term, under the outer clamp only
                        const float hc = ec * sHc[tok];
                        x1 += hc * sKin[d + r];
                        y1 += hc * sKin[DP + d + r];
                    }
                    dq[r] = x1 + 2.0f * q[r] * y1;
                }
                store_out(a.dq, a.dt_g, gbase + static_cast<int64_t>(c * kC + tok) * a.g_sl + d, dq, a.D - d, VEC && a.g_vec);
            }
        }
        __syncthreads();
    }
    if constexpr (DIN) {
        if (a.dsi1) {
            corr += xor_lane<1>(corr);
            corr += xor_lane<2>(corr);
            corr += xor_lane<4>(corr);
            const int f = tid >> 3;
            if ((tid & 7) == 0 && f < K::FP && (f & (DP - 1)) < a.D) {
                if (f < DP) a.kc1[static_cast<size_t>(seq) * a.kc_s + f] = corr;
                else a.kc2[static_cast<size_t>(seq) * a.kc_s + f - DP] = corr;
            }
            if (tid == 0) a.kc0[static_cast<size_t>(seq) * a.kc0_s] = corr0;
        }
    }
    if constexpr (SEL) {
        // <dstate_out, state_out> (the last segment's): the final state's share of the log decays' adjoint
        if (seg == a.G - 1) {
            float fp = 0.f;
            if (a.ds1) {
                const StatePtrs o = seq_state(a.ds0, a.ds1, a.ds2, a.dk0, a.dk1, a.dk2, seq, a.D);
                Carry<DP> X;
                load_carry<DP>(o, a.D, 1.0f, u, g, c16, tid, X);
#pragma unroll
                for (int r = 0; r < 4; ++r) fp += C.m[0][r] * X.m[0][r] + C.m[1][r] * X.m[1][r];
                if ((tid & 7) == 0 && (tid >> 3) < K::FP) fp += C.kf * X.kf;
                if ((tid & 15) == 0 && (tid >> 4) < DP) fp += C.s0 * X.s0;
                if (tid == 0) fp += C.k0 * X.k0;
            }
            fp = wave_sum(fp);
            if (lane == 0) sFin[w] = fp;
            __syncthreads();
            if (tid == 0) {
                float tot = 0.f;
                for (int n = 0; n < kNW; ++n) tot += sFin[n];
                a.fin[seq] = tot;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// dk/dv pass: chunks in reverse, the adjoint of the state leaving each chunk
// carried; it ends as the adjoint of the incoming state.  SEL: also per token
// phi_k'(j) . dphi_k'(j), with the dq pass's query-side terms the log decays'
// adjoint (a suffix sum over the tokens, carried from the last chunk back), and the
// key scale's adjoint per sequence.  DUAL (D = 64): the dual-state pass of a
// segment -- from a zero adjoint, no dk / dv, the adjoint reached at the segment's
// start (its contribution) written to its slot for the reverse scan over segments.
// ---------------------------------------------------------------------------
template <int DP, bool SEL, bool VEC, bool DUAL>
__global__ __launch_bounds__(kT, 1) void chunk_f32_dkv_kernel(const ChunkF32Args a) {
    using K = Dim<DP>;
    __shared__ __attribute__((aligned(16))) float sQ[kC][K::PC];
    __shared__ __attribute__((aligned(16))) float sK[kC][K::PR];
    __shared__ __attribute__((aligned(16))) float sV[kC][K::PR];
    __shared__ __attribute__((aligned(16))) float sG[kC][K::PC];
    __shared__ __attribute__((aligned(16))) float sA[kC][kPAt];     // a, then da
    __shared__ __attribute__((aligned(16))) float sM[K::FP][K::PB];  // dM
    __shared__ float sKf[K::FP], sS0[DP], sPw[kC + 1], sCum[2 * kC], sEc[kC], sW[kC], sH[kC], sEh[kC], sSc[2];
    __shared__ float sPp[K::ND][kC], sPc[kC];  // SEL: the feature blocks' parts, the constant feature's
    __shared__ float sFin[kNW];
    __shared__ int sBad;  // (!VEC) 1 + the last chunk with an infinite or NaN operand

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, c16 = lane & 15;
    const int unit = blockIdx.x;
    const int seq = unit / a.G, seg = unit - seq * a.G;
    const int b = seq / a.H, h = seq - b * a.H;
    const int u = kNW - 1 - w;
    // the adjoint in M's convention: dM = [dS1; 2 dS2], dKf = [dK1; 2 dK2] (the selective
    // convention as it is); a segment's slot holds it so
    const float c2in = SEL ? 1.0f : 2.0f, c2out = SEL ? 1.0f : 0.5f;
    float *slot = a.G > 1 ? a.slots + static_cast<size_t>(unit) * kWsStride : nullptr;
    Carry<DP> C;
    {
        StatePtrs in = seq_state(a.ds0, a.ds1, a.ds2, a.dk0, a.dk1, a.dk2, seq, a.D);
        if (slot) in = slot_state(slot);
        if (DUAL) in.s1 = nullptr;
        load_carry<DP>(in, a.D, slot ? 1.0f : c2in, u, g, c16, tid, C);
    }
    if constexpr (!SEL) put_powers(a, h, tid, sPw);

    const int NC = (a.L + kC - 1) / kC;
    const int c_begin = seg * a.cps, c_end = min(c_begin + a.cps, NC);
    const int i = tid >> 4, part = tid & 15, d0 = K::NE * part;
    const int64_t gbase = b * a.g_sb + h * a.g_sh;
    const int jb = w / K::ND, xb = w % K::ND, tok = 16 * jb + c16;  // this wave's unit of dv and dFk
    // SEL: the suffix sum carried from the last chunk back (wave 0), starting with the final
    // state's share; this thread's part of the key scale's adjoint
    float dl_carry = SEL && !DUAL && seg == a.G - 1 ? a.fin[seq] : 0.f, dks = 0.f;
    Rows<DP> R;
    float inv = 0.f, hd = 0.f;  // the token's 1/D and h
    float seg_ld = 0.f;         // (DUAL, selective, wave 0) the segment's log decay
    auto load = [&](int c) {
        load_rows<DP, VEC, SEL, true>(a, b, h, seq, c, tid, R);
        const size_t o = static_cast<size_t>(seq) * a.L + c * kC;
        const int r = min(i, a.L - c * kC - 1);
        inv = (a.inv_den + o)[r];
        hd = (a.g_den + o)[r];
    };
    load(c_end - 1);
    if constexpr (!VEC) {
        if (tid == 0) sBad = 0;
    }
    if constexpr (!SEL || !VEC) __syncthreads();
    for (int c = c_end - 1; c >= c_begin; --c) {
        const int nv = min(kC, a.L - c * kC);
        float gr[K::NE];
        to_f32<DP, VEC>(R.dy, a.dt_dy, d0, a.D, i < nv, gr);
#pragma unroll
        for (int e = 0; e < K::NE; ++e) gr[e] = i < nv ? gr[e] * inv : 0.f;
        put_elems<DP>(sG, i, d0, gr);
        const float sq = put_rows<DP, VEC, false, 1>(a, R, i, d0, nv, SEL ? a.k_scale[h] : 1.0f, sQ, sK, sV);
        if (!VEC && !(add_squares<DP>(gr, sq) < INFINITY)) sBad = c + 1;
        publish<DP>(C, u, g, c16, tid, sM, sKf, sS0);
        if (part == 0) sH[i] = i < nv ? hd : 0.f;
        if (w == 0) {
            put_decays<SEL>(nv, lane, R.ld, sPw, sCum, sEc, sW, sSc);
            if (SEL && DUAL) seg_ld += wave_sum(lane < nv ? R.ld : 0.f);
        }
        __syncthreads();
        if (c > c_begin) load(c - 1);
        if (tid < kC) sEh[tid] = sEc[tid] * sH[tid];
        const float wj = sW[tok];
        // ---- dv^T tile (value block xb, tokens of block jb): the carried adjoint's part, w_j (Fk_j dM + dS0)
        f32x4 ov = {0.f, 0.f, 0.f, 0.f};
        if constexpr (!DUAL) {
            if (w < 4 * K::ND) {
                f32x4 y = {0.f, 0.f, 0.f, 0.f};
                pipe<4, Op3>(
                    DP / 16,
                    [&](int s) {
                        return Op3{sK[tok][4 * s + g], sM[4 * s + g][16 * xb + c16], sM[DP + 4 * s + g][16 * xb + c16]};
                    },
                    [&](const Op3 &o) {
                        const float wk = wj * o.a;
                        ov = mfma4(o.b, wk, ov);
                        y = mfma4(o.c, 0.5f * (wk * o.a), y);
                    });
#pragma unroll
                for (int r = 0; r < 4; ++r) ov[r] += y[r] + wj * sS0[16 * xb + 4 * g + r];
            }
            if (w < 10) put_scores<DP, SEL>(w, nv, g, c16, sQ, sK, sPw, sCum, sA);
        }
        __syncthreads();
        const float e63 = sSc[0];
        const float k0 = C.k0;  // dK0 of the state leaving the chunk
        f32x4 da = {0.f, 0.f, 0.f, 0.f};
        f32x4 fx = {0.f, 0.f, 0.f, 0.f}, fy = {0.f, 0.f, 0.f, 0.f};
        if constexpr (!DUAL) {
            if (w < 4 * K::ND) {
                // dv: the chunk's part, sum_i a_ij g_i (a_ij = 0 for i < j)
                const bool bad = !VEC && __builtin_amdgcn_readfirstlane(sBad) == c + 1;
                const int i0 = 16 * jb + (bad ? 16 : 0);
                if (i0 < kC)
                    pipe<4, Op2>(
                        4 - i0 / 16, [&](int s) { return Op2{sG[i0 + 4 * s + g][16 * xb + c16], sA[i0 + 4 * s + g][tok]}; },
                        [&](const Op2 &o) { ov = mfma4(o.a, o.b, ov); });
                if (bad) diag_cols(jb, xb, g, tok, sG, sA, ov);
                if (tok < nv) {
                    const int d = 16 * xb + 4 * g;
                    store_out(a.dv, a.dt_g, gbase + static_cast<int64_t>(c * kC + tok) * a.g_sl + d, ov, a.D - d, VEC && a.g_vec);
                }
                // ---- dFk^T tiles (feature block xb and its squares; tokens of block jb): the carried part
                pipe<4, Op3>(
                    DP / 16,
                    [&](int s) {
                        return Op3{sV[tok][4 * s + g], sM[16 * xb + c16][4 * s + g], sM[DP + 16 * xb + c16][4 * s + g]};
                    },
                    [&](const Op3 &o) {
                        const float wv = wj * o.a;
                        fx = mfma4(o.b, wv, fx);
                        fy = mfma4(o.c, wv, fy);
                    });
            }
            if (w < 10) da = dscore_tile<DP, SEL>(w, nv, g, c16, sG, sV, sH, sPw, sCum);
        }
        {
            float sumk = 0.f;
#pragma unroll 8
            for (int t = 0; t < kC; ++t) sumk += sEh[t];
            advance<DP>(C, 1.0f, e63, sumk, u, g, c16, tid, sQ, sG, sEc, sEh);
        }
        __syncthreads();
        if constexpr (!DUAL) {
            if (w < 10) put_tile(w, g, c16, da, sA);
            __syncthreads();
            // ---- dFk: the chunk's part, sum_i da_ij Fq_i -> dk
            if (w < 4 * K::ND) {
                const bool bad = !VEC && __builtin_amdgcn_readfirstlane(sBad) == c + 1;
                const int i0 = 16 * jb + (bad ? 16 : 0);
                if (i0 < kC)
                    pipe<4, Op2>(
                        4 - i0 / 16, [&](int s) { return Op2{sQ[i0 + 4 * s + g][16 * xb + c16], sA[i0 + 4 * s + g][tok]}; },
                        [&](const Op2 &o) {
                            fx = mfma4(o.a, o.b, fx);
                            fy = mfma4(o.a * o.a, o.b, fy);
                        });
                if (bad) {
                    diag_cols(jb, xb, g, tok, sQ, sA, fx);
                    for (int j = tok; j < 16 * jb + 16; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float q = sQ[j][16 * xb + 4 * g + r];
                            fy[r] = fmaf(q * q, sA[j][tok], fy[r]);
                        }
                }
                const int d = 16 * xb + 4 * g;
                const f32x4 k = ld4(&sK[tok][d]);
                f32x4 dk;
                float pkp = 0.f;  // SEL: sum over this lane's features of Fk . dFk
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x1 = fx[r] + wj * sKf[d + r], y1 = fy[r] + wj * sKf[DP + d + r];
                    dk[r] = x1 + k[r] * y1;
                    if constexpr (SEL) pkp += k[r] * x1 + 0.5f * (k[r] * k[r]) * y1;
                }
                if constexpr (SEL) {
                    pkp = sum_lane32(sum_lane16(pkp));
                    if (g == 0) sPp[xb][tok] = pkp;
                    // k is kscale times the key: dk above is the scaled key's adjoint; the key's is
                    // kscale times it, the scale's the sum over the key's elements of it (below, from LDS)
                }
                if (tok < nv) {
                    if constexpr (SEL) {
                        const float ks = a.k_scale[h];
                        const void *kp = static_cast<const char *>(a.k) +
                                         (b * a.k_sb + (h / a.group) * a.k_sh + static_cast<int64_t>(c) * kC * a.k_sl) *
                                             (a.dt_k == PRIME_F32 ? 4 : 2);
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (d + r < a.D) dks += load_elem(kp, min(tok, nv - 1) * a.k_sl + d + r, a.dt_k) * dk[r];
                            dk[r] *= ks;
                        }
                    }
                    store_out(a.dk, a.dt_g, gbase + static_cast<int64_t>(c * kC + tok) * a.g_sl + d, dk, a.D - d, VEC && a.g_vec);
                }
            }
            if constexpr (SEL) {
                // the constant feature: sum_i da_ij + w_j (dS0 . v_j + dK0), of the adjoint leaving the chunk
                // (16 threads a token; only da's lower tiles exist)
                float cs = 0.f, vs = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e >= (i >> 4)) cs += sA[16 * e + part][i];
#pragma unroll
                for (int e = 0; e < K::NE; ++e) vs += sS0[d0 + e] * sV[i][d0 + e];
                cs = sum16(cs + sW[i] * vs) + sW[i] * k0;
                if (part == 0) sPc[i] = cs;
            }
            __syncthreads();
            if constexpr (SEL) {
                // the log decays' adjoint: per token dc = phi_q' . dphi_q' - phi_k' . dphi_k', summed over
                // every later token (a suffix sum over the chunk, plus the carry)
                if (w == 0) {
                    const size_t t = static_cast<size_t>(seq) * a.L + c * kC + lane;
                    float x = 0.f;
                    if (lane < nv) {
                        x = a.pq[t] - sPc[lane];
#pragma unroll
                        for (int n = 0; n < K::ND; ++n) x -= sPp[n][lane];
                    }
                    const float pre = wave_prefix_sum(x);
                    const float tot = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pre), 63));
                    if (lane < nv) a.dlogd[t] = tot - pre + x + dl_carry;
                    dl_carry += tot;
                }
            }
        }
    }
    if constexpr (DUAL) {
        store_carry<DP>(slot_state(slot), a.D, 1.0f, u, g, c16, tid, C);
        if (SEL && tid == 0) slot[kWsDecay] = seg_ld * 1.44269504088896341f;  // log2
        return;
    }
    if constexpr (SEL) {  // the key scale's adjoint, this unit's share; the segment's suffix total
        const float v = wave_sum(dks);
        if (lane == 0) sFin[w] = v;
        __syncthreads();
        if (tid == 0) {
            float tot = 0.f;
            for (int n = 0; n < kNW; ++n) tot += sFin[n];
            if (a.G == 1) {
                a.dkscale[seq] = tot;
            } else {
                a.seg_tot[2 * unit] = dl_carry;
                a.seg_tot[2 * unit + 1] = tot;
            }
        }
    }
    // ---- adjoint of the incoming state (with segments the reverse scan over them writes it)
    if (a.dsi1 && a.G == 1) {
        const StatePtrs o = seq_state(a.dsi0, a.dsi1, a.dsi2, a.dki0, a.dki1, a.dki2, seq, a.D);
        if (a.dense_clamp && a.s1i) {
            // plus the dq pass's correction (features [K1; K2/2], K0)
            const int f = tid >> 3;
            const size_t kc = static_cast<size_t>(seq) * a.kc_s;
            if (f < K::FP && (f & (DP - 1)) < a.D) C.kf += f < DP ? a.kc1[kc + f] : a.kc2[kc + f - DP];
            C.k0 += a.kc0[static_cast<size_t>(seq) * a.kc0_s];
            __syncthreads();  // (before any of them is written)
        }
        store_carry<DP>(o, a.D, c2out, u, g, c16, tid, C);
    }
}

namespace {

template <int DP, bool VEC>
void launch_prefill_dp(const ChunkF32Args &a, dim3 grid, hipStream_t s, const TimerEvents &t) {
    const dim3 block(kT);
    if (a.selective)
        hipExtLaunchKernelGGL((chunk_f32_prefill_kernel<DP, false, true, VEC, false>), grid, block, 0, s, t.start, t.stop,
                              0, a);
    else if (a.dense_clamp && a.s1i)
        hipExtLaunchKernelGGL((chunk_f32_prefill_kernel<DP, true, false, VEC, false>), grid, block, 0, s, t.start, t.stop,
                              0, a);
    else
        hipExtLaunchKernelGGL((chunk_f32_prefill_kernel<DP, false, false, VEC, false>), grid, block, 0, s, t.start,
                              t.stop, 0, a);
}

template <int DP, bool VEC>
void launch_dq_dp(const ChunkF32Args &a, dim3 grid, hipStream_t s, const TimerEvents &t) {
    const dim3 block(kT);
    if (a.selective)
        hipExtLaunchKernelGGL((chunk_f32_dq_kernel<DP, false, true, VEC>), grid, block, 0, s, t.start, t.stop, 0, a);
    else if (a.dense_clamp && a.s1i)
        hipExtLaunchKernelGGL((chunk_f32_dq_kernel<DP, true, false, VEC>), grid, block, 0, s, t.start, t.stop, 0, a);
    else
        hipExtLaunchKernelGGL((chunk_f32_dq_kernel<DP, false, false, VEC>), grid, block, 0, s, t.start, t.stop, 0, a);
}

template <int DP, bool VEC>
void launch_dkv_dp(const ChunkF32Args &a, dim3 grid, hipStream_t s, const TimerEvents &t) {
    const dim3 block(kT);
    if (a.selective)
        hipExtLaunchKernelGGL((chunk_f32_dkv_kernel<DP, true, VEC, false>), grid, block, 0, s, t.start, t.stop, 0, a);
    else
        hipExtLaunchKernelGGL((chunk_f32_dkv_kernel<DP, false, VEC, false>), grid, block, 0, s, t.start, t.stop, 0, a);
}

}  // namespace

// Selective backward in segments: each segment's dk/dv pass left the suffix sums of
// its own tokens and its totals; every token gets the later segments' totals added,
// and the key scale's adjoint is summed over the segments.  One workgroup a sequence.
__global__ __launch_bounds__(256) void chunk_f32_seg_totals_kernel(const ChunkF32Args a) {
    const int seq = blockIdx.x;
    const float *tot = a.seg_tot + static_cast<size_t>(seq) * a.G * 2;
    float ks = 0.f;
    for (int s = 0; s < a.G; ++s) ks += tot[2 * s + 1];
    if (threadIdx.x == 0) a.dkscale[seq] = ks;
    const int T = a.cps * kC;
    float carry = 0.f;
    for (int s = a.G - 2; s >= 0; --s) {
        carry += tot[2 * (s + 1)];
        for (int t = s * T + threadIdx.x; t < (s + 1) * T; t += 256) a.dlogd[static_cast<size_t>(seq) * a.L + t] += carry;
    }
}

hipError_t launch_chunk_f32_prefill(const ChunkF32Args &a, hipStream_t stream) {
    const TimerEvents t = timer_events(PRIME_KERNEL_PREFILL_CHUNKS);
    const dim3 grid(a.B * a.H * a.G);
    if (a.D <= 16) launch_prefill_dp<16, false>(a, grid, stream, t);
    else if (a.D <= 32) launch_prefill_dp<32, false>(a, grid, stream, t);
    else launch_prefill_dp<64, false>(a, grid, stream, t);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) timer_drop(t);
    return e;
}

hipError_t launch_chunk_f32_backward(const ChunkF32Args &a, hipStream_t stream) {
    const dim3 grid(a.B * a.H * a.G);
    hipError_t e;
    const TimerEvents t1 = timer_events(PRIME_KERNEL_BWD_DQ);
    if (a.D <= 16) launch_dq_dp<16, false>(a, grid, stream, t1);
    else if (a.D <= 32) launch_dq_dp<32, false>(a, grid, stream, t1);
    else launch_dq_dp<64, false>(a, grid, stream, t1);
    if ((e = hipGetLastError()) != hipSuccess) return timer_drop(t1), e;
    const TimerEvents t2 = timer_events(PRIME_KERNEL_BWD_DKV);
    if (a.D <= 16) launch_dkv_dp<16, false>(a, grid, stream, t2);
    else if (a.D <= 32) launch_dkv_dp<32, false>(a, grid, stream, t2);
    else launch_dkv_dp<64, false>(a, grid, stream, t2);
    if ((e = hipGetLastError()) != hipSuccess) timer_drop(t2);
    return e;
}

// ---------------------------------------------------------------------------
// D = 64, fp32 rows on 16-byte boundaries: selective PRIME's prefill and both
// backwards, few long sequences in segments.
// ---------------------------------------------------------------------------
namespace {

template <class A>
void copy_common(ChunkF32Args &o, const A &a) {
    o.q = a.q; o.k = a.k; o.v = a.v;
    o.q_sb = a.q_sb; o.q_sh = a.q_sh; o.q_sl = a.q_sl;
    o.k_sb = a.k_sb; o.k_sh = a.k_sh; o.k_sl = a.k_sl;
    o.v_sb = a.v_sb; o.v_sh = a.v_sh; o.v_sl = a.v_sl;
    o.dt_q = o.dt_k = o.dt_v = a.dt_in;
    o.B = a.B; o.H = a.H; o.L = a.L; o.D = kD; o.group = 1;
    o.decay = a.decay; o.eps = a.eps;
    o.s0i = a.s0i; o.s1i = a.s1i; o.s2i = a.s2i; o.k0i = a.k0i; o.k1i = a.k1i; o.k2i = a.k2i;
    o.G = a.G; o.cps = a.cps; o.slots = a.ws;
}

// every segment's state from zero, then the state entering each
hipError_t launch_segment_states(const ChunkF32Args &o, const PrefillArgs &p, hipStream_t stream) {
    const TimerEvents ta = timer_events(PRIME_KERNEL_PREFILL_SEGMENTS);
    const dim3 grid(o.B * o.H * (o.G - 1));
    if (o.selective)
        hipExtLaunchKernelGGL((chunk_f32_prefill_kernel<64, false, true, true, true>), grid, dim3(kT), 0, stream,
                              ta.start, ta.stop, 0, o);
    else
        hipExtLaunchKernelGGL((chunk_f32_prefill_kernel<64, false, false, true, true>), grid, dim3(kT), 0, stream,
                              ta.start, ta.stop, 0, o);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return timer_drop(ta), e;
    return launch_segment_scan(p, stream);
}

}  // namespace

hipError_t launch_selective_f32(const PrefillArgs &a, hipStream_t stream) {
    ChunkF32Args o{};
    copy_common(o, a);
    o.group = a.group;
    o.selective = 1;
    o.log_decay = a.log_decay; o.k_scale = a.k_scale;
    o.s0o = a.s0o; o.s1o = a.s1o; o.s2o = a.s2o; o.k0o = a.k0o; o.k1o = a.k1o; o.k2o = a.k2o;
    o.y = a.y; o.dt_y = a.dt_y; o.y_sb = a.y_sb; o.y_sh = a.y_sh; o.y_sl = a.y_sl;
    hipError_t e;
    if (a.G > 1 && (e = launch_segment_states(o, a, stream)) != hipSuccess) return e;
    const TimerEvents t = timer_events(PRIME_KERNEL_PREFILL_CHUNKS);
    hipExtLaunchKernelGGL((chunk_f32_prefill_kernel<64, false, true, true, false>), dim3(a.B * a.H * a.G), dim3(kT), 0,
                          stream, t.start, t.stop, 0, o);
    if ((e = hipGetLastError()) != hipSuccess) timer_drop(t);
    return e;
}

hipError_t launch_prefill_backward_f32(const BwdArgs &a, hipStream_t stream) {
    ChunkF32Args o{};
    copy_common(o, a);
    const bool sel = a.logd != nullptr;
    o.selective = sel;
    o.log_decay = a.logd; o.k_scale = a.kscale;
    o.dense_clamp = a.dense_in;
    o.dy = a.dy; o.dt_dy = a.dt_dy; o.dy_sb = a.dy_sb; o.dy_sh = a.dy_sh; o.dy_sl = a.dy_sl;
    o.ds0 = a.ds0o; o.ds1 = a.ds1o; o.ds2 = a.ds2o; o.dk0 = a.dk0o; o.dk1 = a.dk1o; o.dk2 = a.dk2o;
    o.dsi0 = a.ds0i; o.dsi1 = a.ds1i; o.dsi2 = a.ds2i; o.dki0 = a.dk0i; o.dki1 = a.dk1i; o.dki2 = a.dk2i;
    o.dq = a.dq; o.dk = a.dk; o.dv = a.dv; o.dt_g = a.dt_g; o.g_sb = a.g_sb; o.g_sh = a.g_sh; o.g_sl = a.g_sl;
    o.g_vec = gradient_rows_vec(a);
    o.inv_den = a.inv_den; o.g_den = a.g_den;
    o.kc1 = a.kcorr; o.kc2 = a.kcorr + kD; o.kc0 = a.kcorr + 2 * kD;
    o.kc_s = o.kc0_s = kBwdCorr;
    o.dlogd = a.dlogd; o.dkscale = a.dkscale; o.pq = a.pq; o.fin = a.fin; o.seg_tot = a.seg_tot;
    const dim3 grid(a.B * a.H * a.G), block(kT);
    hipError_t e;
    if (a.G > 1) {
        // (in fp32: the states of the prefill's own state-only pass, formed from operands split
        // into two bf16 parts, put dq 4e-6 from float64 at 8 segments, against 9e-7)
        PrefillArgs p{};
        p.B = a.B; p.H = a.H; p.group = 1; p.L = a.L; p.G = a.G; p.cps = a.cps; p.ws = a.ws;
        p.decay = a.decay; p.log_decay = a.logd;
        p.s0i = a.s0i; p.s1i = a.s1i; p.s2i = a.s2i; p.k0i = a.k0i; p.k1i = a.k1i; p.k2i = a.k2i;
        if ((e = launch_segment_states(o, p, stream)) != hipSuccess) return e;
    }
    const TimerEvents t1 = timer_events(PRIME_KERNEL_BWD_DQ);
    launch_dq_dp<64, true>(o, grid, stream, t1);
    if ((e = hipGetLastError()) != hipSuccess) return timer_drop(t1), e;
    if (a.G > 1) {
        // each segment's dual contribution, then the reverse scan (slots now hold dual states)
        const TimerEvents td = timer_events(PRIME_KERNEL_BWD_DUAL);
        if (sel)
            hipExtLaunchKernelGGL((chunk_f32_dkv_kernel<64, true, true, true>), grid, block, 0, stream, td.start, td.stop,
                                  0, o);
        else
            hipExtLaunchKernelGGL((chunk_f32_dkv_kernel<64, false, true, true>), grid, block, 0, stream, td.start,
                                  td.stop, 0, o);
        if ((e = hipGetLastError()) != hipSuccess) return timer_drop(td), e;
        if ((e = launch_bwd_dual_scan(a, stream)) != hipSuccess) return e;
    }
    const TimerEvents t2 = timer_events(PRIME_KERNEL_BWD_DKV);
    launch_dkv_dp<64, true>(o, grid, stream, t2);
    if ((e = hipGetLastError()) != hipSuccess) return timer_drop(t2), e;
    if (sel && a.G > 1) {
        hipLaunchKernelGGL(chunk_f32_seg_totals_kernel, dim3(a.B * a.H), dim3(256), 0, stream, o);
        e = hipGetLastError();
    }
    return e;
}

}  // namespace prime
