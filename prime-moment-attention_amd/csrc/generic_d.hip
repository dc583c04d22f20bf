// PRIME moment attention for head dims other than 64 (D < 64), token by token: the
// decode step (attention.py:119-143 at any head_dim, as the reference's own
// tests run it at head_dim 32, tests/test_attention.py:7-14) and calls of a few
// tokens on many sequences, the base and the selective form; and
// prime_head_layernorm for these dims.  Other calls of several tokens run the
// chunked kernels (chunk_f32.hip).
//
// One wavefront per (sequence, head): lane j < D owns value column j of the
// state -- S0[j], S1[:, j], S2[:, j] in registers -- and lane D the "ones"
// column that carries the normaliser K0, K1, K2 (the moments of a value that
// is always 1), so one readout gives every lane its numerator and lane D the
// denominator:
//   S <- l S + k v^T (v_D = 1),  num_j = S0_j + q . S1[:, j] + 1/2 q^2 . S2[:, j]
//   y_j = num_j / max(num_D, eps)
// (the update before the readout, attention.py:126-143).  Lanes read q and k
// from LDS, where the token is staged (and, with a QK LayerNorm, normalised on
// load).  The dense branch's double clamp (attention.py:177-185, with an
// incoming state) splits the denominator into the call's part and the incoming
// state's readout of its K moments (held in LDS).
// fp32 arithmetic; bf16 / fp16 / fp32 storage.

#include <algorithm>

#include "head_row.h"
#include "prime_kernels.h"

namespace prime {
namespace {

constexpr int kGD = 64;     // lanes: value columns 0 .. D-1 and the ones column D (D < 64)
constexpr int kGC = 64;     // rows per workgroup of the head LayerNorm
constexpr int kGP = kGD + 1;

}  // namespace

// MULTI: a.L tokens in order, else one.
template <bool MULTI>
__global__ __launch_bounds__(kGD) void generic_step_kernel(const GenericArgs a) {
    __shared__ float sq[kGP], sk[kGP], sdec[1];
    __shared__ float sKin[3][kGP];  // incoming K1, K2 (dense clamp), K0 at [2][0]
    const int lane = threadIdx.x, bh = blockIdx.x;
    const int b = bh / a.H, h = bh - b * a.H, hk = h / a.group, D = a.D;
    const bool col = lane <= D;
    const bool sel = a.selective != 0;
    // the second-order weights: k*k and q*q/2 (base), (beta k)*(beta k)/2 and q*q (selective)
    const float ck2 = sel ? 0.5f : 1.0f, cq2 = sel ? 1.0f : 0.5f;
    const size_t o1 = static_cast<size_t>(bh) * D * D, o0 = static_cast<size_t>(bh) * D;
    // ---- a token: q and k for LDS, v in its lane
    float qx, kx, vx;
    auto load_token = [&](int t) {
        qx = lane < D ? load_elem(a.q, b * a.q_sb + h * a.q_sh + t * a.q_sl + lane, a.dt_q) : 0.f;
        kx = lane < D ? load_elem(a.k, b * a.k_sb + hk * a.k_sh + t * a.k_sl + lane, a.dt_k) : 0.f;
        vx = lane < D ? load_elem(a.v, b * a.v_sb + hk * a.v_sh + t * a.v_sl + lane, a.dt_v) : (lane == D ? 1.0f : 0.0f);
    };
    load_token(0);
    sq[lane] = qx;
    sk[lane] = kx;
    float S0 = 0.f, S1[kGD - 1], S2[kGD - 1];
#pragma unroll
    for (int i = 0; i < kGD - 1; ++i) {
        S1[i] = S2[i] = 0.f;
        if (i < D && col && a.s1i) {
            S1[i] = lane < D ? a.s1i[o1 + i * D + lane] : a.k1i[o0 + i];
            S2[i] = lane < D ? a.s2i[o1 + i * D + lane] : a.k2i[o0 + i];
        }
    }
    if (col && a.s1i) S0 = lane < D ? a.s0i[o0 + lane] : a.k0i[bh];
    const bool dense = a.dense_clamp && a.s1i;
    if (dense) {
        if (lane < D) {
            sKin[0][lane] = a.k1i[o0 + lane];
            sKin[1][lane] = a.k2i[o0 + lane];
        }
        if (lane == 0) sKin[2][0] = a.k0i[bh];
    }
    float lin = 1.f;  // the incoming state's decay
    for (int t = 0; t < (MULTI ? a.L : 1); ++t) {
        if (MULTI && t) {
            __syncthreads();  // (the last token's reads)
            sq[lane] = qx;
            sk[lane] = kx;
        }
        const float vj = vx;
        if (MULTI && t + 1 < a.L) load_token(t + 1);
        __syncthreads();
        if (a.qk_norm) {
            if (lane == 0) generic_ln_row(sq, D, a.qn_w, a.qn_b, a.dt_norm, a.ln_eps, a.q_scale, a.dt_q);
            if (lane == 1) generic_ln_row(sk, D, a.kn_w, a.kn_b, a.dt_norm, a.ln_eps, 1.0f, a.dt_k);
            __syncthreads();
        }
        if (sel) {
            sk[lane] *= a.k_scale[h];
            if (lane == 0) {
                float lam_t;
                if (a.log_decay) {
                    lam_t = expf(a.log_decay[MULTI ? static_cast<size_t>(bh) * a.L + t : bh]);
                } else if (a.decay_bh) {
                    lam_t = a.decay_bh[bh];
                } else {
                    // selective.py:368, 386: Delta = clamp(softplus(s)), each stage
                    // rounded to the step's dtype as the module's tensors are
                    const float sv0 = load_elem(a.step, b * a.step_sb + h, a.dt_step);
                    float d = sv0 > 20.f ? sv0 : log1pf(expf(sv0));
                    d = round_dt(d, a.dt_step);
                    d = round_dt(fminf(fmaxf(d, a.step_min), a.step_max), a.dt_step);
                    lam_t = expf(-d / a.tau[h]);
                }
                sdec[0] = lam_t;
            }
            __syncthreads();
        }
        const float lt = sel ? sdec[0] : a.decay[h];
        S0 = lt * S0 + vj;
        float num = S0;
#pragma unroll
        for (int i = 0; i < kGD - 1; ++i) {
            if (i < D) {
                const float ki = sk[i], qi = sq[i];
                S1[i] = fmaf(lt, S1[i], ki * vj);
                S2[i] = fmaf(lt, S2[i], ck2 * ki * ki * vj);
                num = fmaf(qi, S1[i], num);
                num = fmaf(cq2 * qi * qi, S2[i], num);
            }
        }
        const float den = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(num), D));
        float den_c;
        if (dense) {
            lin *= lt;
            float di = sKin[2][0];
            for (int i = 0; i < D; ++i) {
                const float qi = sq[i];
                di = fmaf(qi, sKin[0][i], di);
                di = fmaf(0.5f * qi * qi, sKin[1][i], di);
            }
            di *= lin;
            den_c = fmaxf(fmaxf(den - di, a.eps) + di, a.eps);
        } else {
            den_c = fmaxf(den, a.eps);
        }
        if (lane < D && a.y)
            store_elem(a.y, b * a.y_sb + h * a.y_sh + (MULTI ? t * a.y_sl : 0) + lane, a.dt_y, num / den_c);
    }
    if (a.s1o && col) {
#pragma unroll
        for (int i = 0; i < kGD - 1; ++i) {
            if (i < D) {
                if (lane < D) {
                    a.s1o[o1 + i * D + lane] = S1[i];
                    a.s2o[o1 + i * D + lane] = S2[i];
                } else {
                    a.k1o[o0 + i] = S1[i];
                    a.k2o[o0 + i] = S2[i];
                }
            }
        }
        if (lane < D) a.s0o[o0 + lane] = S0;
        else a.k0o[bh] = S0;
    }
}

// Few tokens on many sequences go token by token: a chunk costs its workgroup the same for
// 2 tokens as for 64, and with several workgroups a CU those add up.  With s sequences a CU
// the line lies at s + 1 tokens, 12 at most: at D = 32 with states, the times of the token
// kernel over the chunk kernel are 1.00 at s = 3 and 4 tokens (1.28 at 2 sequences and 3
// tokens), 0.84 at 4 and 4 (1.02 at 6 tokens), 0.86 at 16 and 12 (1.07 at 16); at D = 48 0.79,
// 0.66 and 0.65.  A QK LayerNorm on load is one lane's work per token here and one lane a
// token there: (s + 1) / 2 tokens, 5 at most (D = 32: 0.98 at 3 and 2, 0.79 at 4 and 2 and 1.09
// at 3, 0.75 at 8 and 4, 0.89 at 16 and 5 and 1.04 at 6).  16,384 sequences of 2 tokens: 608 us in
// chunks, 204 token by token (D = 32); 4096 of 2 at D = 48 236 and 65.
static bool token_by_token(const GenericArgs &a) {
    const int64_t s = static_cast<int64_t>(a.B) * a.H / device_cus();
    return s >= 3 && a.L <= (a.qk_norm ? std::min<int64_t>((s + 1) / 2, 5) : std::min<int64_t>(s + 1, 12));
}

hipError_t launch_generic_prefill(GenericArgs a, hipStream_t stream) {
    const dim3 grid(a.B * a.H), block(kGD);
    if (a.L == 1) hipLaunchKernelGGL(generic_step_kernel<false>, grid, block, 0, stream, a);
    else if (token_by_token(a)) hipLaunchKernelGGL(generic_step_kernel<true>, grid, block, 0, stream, a);
    else return launch_chunk_f32_prefill(a, stream);
    return hipGetLastError();
}

// prime_head_layernorm for head dims below 64: 64 rows per wavefront, staged
// through LDS with coalesced loads, lane r normalising row r.
__global__ __launch_bounds__(kGD) void generic_head_layernorm_kernel(const HeadNormArgs a) {
    __shared__ float rows[kGC][kGP];
    const int lane = threadIdx.x, D = a.D;
    const int64_t nrows = static_cast<int64_t>(a.B) * a.H * a.L, r0 = static_cast<int64_t>(blockIdx.x) * kGC;
    const int nv = static_cast<int>(min(static_cast<int64_t>(kGC), nrows - r0));
    auto offs = [&](int t, int64_t sb, int64_t sh, int64_t sl) {
        const int64_t r = r0 + t, h = r % a.H, bl = r / a.H, l = bl % a.L, b = bl / a.L;
        return b * sb + h * sh + l * sl;
    };
    for (int t = 0; t < nv; ++t)
        rows[t][lane] = lane < D ? load_elem(a.x, offs(t, a.x_sb, a.x_sh, a.x_sl) + lane, a.dt) : 0.f;
    __syncthreads();
    if (lane < nv) generic_ln_row(rows[lane], D, a.weight, a.bias, a.dt_norm, a.ln_eps, a.scale, a.dt);
    __syncthreads();
    for (int t = 0; t < nv; ++t)
        if (lane < D) store_elem(a.out, offs(t, a.o_sb, a.o_sh, a.o_sl) + lane, a.dt, rows[t][lane]);
}

hipError_t launch_generic_head_layernorm(const HeadNormArgs &a, hipStream_t stream) {
    const int64_t rows = static_cast<int64_t>(a.B) * a.H * a.L;
    hipLaunchKernelGGL(generic_head_layernorm_kernel, dim3(static_cast<uint32_t>((rows + kGC - 1) / kGC)),
                       dim3(kGD), 0, stream, a);
    return hipGetLastError();
}

}  // namespace prime
