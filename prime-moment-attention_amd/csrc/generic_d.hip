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
constexpr int kFew = 16;    // tokens of a call that goes token by token, at most

}  // namespace

// T: tokens staged (one, or up to T = kFew of a call), taken in order.
template <int T>
__global__ __launch_bounds__(kGD) void generic_step_kernel(const GenericArgs a) {
    __shared__ float sq[T][kGP], sk[T][kGP], sv[T][kGP], sdec[T];
    __shared__ float sKin[3][kGP];  // incoming K1, K2 (dense clamp), K0 at [2][0]
    const int lane = threadIdx.x, bh = blockIdx.x;
    const int b = bh / a.H, h = bh - b * a.H, hk = h / a.group, D = a.D;
    const int L = T == 1 ? 1 : a.L;
    const bool col = lane <= D;
    const bool sel = a.selective != 0;
    // the second-order weights: k*k and q*q/2 (base), (beta k)*(beta k)/2 and q*q (selective)
    const float ck2 = sel ? 0.5f : 1.0f, cq2 = sel ? 1.0f : 0.5f;
    const size_t o1 = static_cast<size_t>(bh) * D * D, o0 = static_cast<size_t>(bh) * D;
    // ---- the tokens' rows in LDS, v with the ones column
    {
        const int64_t qo = b * a.q_sb + h * a.q_sh + lane, ko = b * a.k_sb + hk * a.k_sh + lane,
                      vo = b * a.v_sb + hk * a.v_sh + lane;
#pragma unroll 4
        for (int t = 0; t < L; ++t) {
            sq[t][lane] = lane < D ? load_elem(a.q, qo + t * a.q_sl, a.dt_q) : 0.f;
            sk[t][lane] = lane < D ? load_elem(a.k, ko + t * a.k_sl, a.dt_k) : 0.f;
            sv[t][lane] = lane < D ? load_elem(a.v, vo + t * a.v_sl, a.dt_v) : (lane == D ? 1.0f : 0.0f);
        }
    }
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
    __syncthreads();
    if (a.qk_norm) {  // a row per lane
        const int t = lane & 31;
        if (t < L) {
            if (lane < 32) generic_ln_row(sq[t], D, a.qn_w, a.qn_b, a.dt_norm, a.ln_eps, a.q_scale, a.dt_q);
            else generic_ln_row(sk[t], D, a.kn_w, a.kn_b, a.dt_norm, a.ln_eps, 1.0f, a.dt_k);
        }
        __syncthreads();
    }
    if (sel) {
        const float ks = a.k_scale[h];
        for (int t = 0; t < L; ++t) sk[t][lane] *= ks;
        if (lane < L) {
            float lam_t;
            if (a.log_decay) {
                lam_t = expf(a.log_decay[static_cast<size_t>(bh) * L + lane]);
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
            sdec[lane] = lam_t;
        }
        __syncthreads();
    }
    const float lh = sel ? 0.f : a.decay[h];
    float lin = 1.f;  // the incoming state's decay
    for (int t = 0; t < L; ++t) {
        const float lt = sel ? sdec[t] : lh, vj = sv[t][lane];
        S0 = lt * S0 + vj;
        float num = S0;
#pragma unroll
        for (int i = 0; i < kGD - 1; ++i) {
            if (i < D) {
                const float ki = sk[t][i], qi = sq[t][i];
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
                const float qi = sq[t][i];
                di = fmaf(qi, sKin[0][i], di);
                di = fmaf(0.5f * qi * qi, sKin[1][i], di);
            }
            di *= lin;
            den_c = fmaxf(fmaxf(den - di, a.eps) + di, a.eps);
        } else {
            den_c = fmaxf(den, a.eps);
        }
        if (lane < D && a.y)
            store_elem(a.y, b * a.y_sb + h * a.y_sh + (T == 1 ? 0 : t * a.y_sl) + lane, a.dt_y, num / den_c);
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
// 2 tokens as for 64, and the chunk kernel runs r = ceil(sequences / CUs) rounds of them.  The
// lines (tokens up to which this kernel was the faster one, at head dims 8 to 63 and 64 to 8192
// sequences) by what a call carries:
//   no state in or out   2 r - 1  from r = 2 (D = 32, r = 2: 15.1 us against 17.1 at 3 tokens, 18.5 at 4);
//                        above D = 32, whose chunks cost more, 3 r - 3
//   states               2 r - 2  from r = 3, 14 at most (D = 32, r = 3: 28.3 against 29.2 at 4, 34.7 at 6)
//   the dense clamp's    2 r - 4, 10 at most (the incoming denominator is read once per token)
//   a QK LayerNorm on load, whose serial row each lane does once here and there:
//                        4 r - 4, with states 4 r - 6, with the dense clamp's 4 r - 8 and 10 at most
// 8192 sequences of 2 tokens at D = 32: 294 us in chunks, 81 token by token; 600 of 2 at D = 48
// without states 40 and 13.
static bool token_by_token(const GenericArgs &a) {
    const int64_t cus = device_cus(), r = (static_cast<int64_t>(a.B) * a.H + cus - 1) / cus;
    const bool state = a.s1i || a.s1o, dense = a.dense_clamp && a.s1i;
    const int64_t line = a.qk_norm ? 4 * r - (dense ? 8 : state ? 6 : 4)
                         : dense   ? 2 * r - 4
                         : state   ? (r < 3 ? 0 : 2 * r - 2)
                                   : (a.D > 32 ? 3 * r - 3 : 2 * r - 1);
    return a.L <= std::min<int64_t>(line, dense ? 10 : state && !a.qk_norm ? 14 : kFew);
}

hipError_t launch_generic_prefill(GenericArgs a, hipStream_t stream) {
    const dim3 grid(a.B * a.H), block(kGD);
    if (a.L == 1) hipLaunchKernelGGL(generic_step_kernel<1>, grid, block, 0, stream, a);
    else if (token_by_token(a)) hipLaunchKernelGGL(generic_step_kernel<kFew>, grid, block, 0, stream, a);
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
