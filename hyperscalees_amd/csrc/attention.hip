// attention.hip -- the spiking self-attention transformer's own kernels (C4).
//
// Model: src/hyperscalees/models/snn_self_attention_heads.py (LIF-encoded
// Q/K/V, multi-head attention whose row weights come from a LIF competition,
// row_softmax_lif of snn_self_attention.py:45-80, a LIF-gated feed-forward
// and a pooled readout).  The perturbed projections run on the forward
// kernels of linear*.hip; these kernels cover what lies between them, batched
// over the population: member m owns rows [m R, (m+1) R) of every (rows, C)
// plane (R = tokens per member).  Thresholds, beta and gains are per-member
// device arrays (the member's perturbed Parameter leaves after softplus).
// All arithmetic is f32 in the reference's operation order; reductions of
// spike counts are exact (integers), the attention dot products and A @ V
// sum in index order.
#include "runtime.h"

namespace hses {

namespace {

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Reduction over the 64 lanes of a wave, the result in every lane: within
// rows of 16 lanes by DPP (quad swaps, then the half-row and row mirrors),
// across rows by the permlane16 and permlane32 swaps (no LDS round trips).
// Callers reduce values whose result does not depend on the order (integer
// counts, maxima).
template <class Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
    v = op(v, dpp_mov<0xB1>(v));   // quad_perm 1,0,3,2
    v = op(v, dpp_mov<0x4E>(v));   // quad_perm 2,3,0,1
    v = op(v, dpp_mov<0x141>(v));  // row_half_mirror
    v = op(v, dpp_mov<0x140>(v));  // row_mirror
    const uint32_t u = __float_as_uint(v);
    const auto p16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = op(__uint_as_float(p16[0]), __uint_as_float(p16[1]));
    const uint32_t w = __float_as_uint(v);
    const auto p32 = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return op(__uint_as_float(p32[0]), __uint_as_float(p32[1]));
}

__device__ __forceinline__ float wsum(float v) {
    return wave_reduce(v, [](float x, float y) { return x + y; });
}

__device__ __forceinline__ float wmax(float v) {
    return wave_reduce(v, [](float x, float y) { return fmaxf(x, y); });
}

// snn_attention.py:41-49 (dt = 1): v + leak * (-v + cur); spike = v >= vth;
// v * (1 - spike).
__device__ __forceinline__ float lif_upd(float v, float cur, float leak, float vth, float* s) {
    const float vn = __fadd_rn(v, __fmul_rn(leak, __fadd_rn(-v, cur)));
    const float sp = vn >= vth ? 1.0f : 0.0f;
    *s = sp;
    return __fmul_rn(vn, __fsub_rn(1.0f, sp));
}

}  // namespace

// jax.nn.softplus = logaddexp(x, 0) = max(x, 0) + log1p(exp(-|x|)).
__global__ __launch_bounds__(256) void k_softplus(const float* __restrict__ x, int64_t n,
                                                  float* __restrict__ y) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) {
        const float v = x[e];
        y[e] = __fadd_rn(fmaxf(v, 0.0f), log1pf(expf(-fabsf(v))));
    }
}

// _rate of the three encoders and their mean plus the position embedding
// (snn_self_attention_heads.py:33-40, 168-175): one thread per row and VEC columns.
// th_q, th_k, th_v: (n) thresholds; pos: (R, d) shared or (n, R, d).
// Bound by its 3 T reads: VEC = 4 where every plane's rows are 16-byte aligned, with
// the three encoders' loads of four steps in flight.
// 1024 members x 64 tokens x 64, T = 8: 149 -> 92 us (2.9 -> 4.7 TB/s; a copy reaches 4.76).
template <int VEC>
__global__ __launch_bounds__(256) void k_sa_encode(const float* __restrict__ cq,
                                                   const float* __restrict__ ck,
                                                   const float* __restrict__ cv, int32_t T,
                                                   int64_t M, int32_t d, int32_t R,
                                                   const float* __restrict__ th_q,
                                                   const float* __restrict__ th_k,
                                                   const float* __restrict__ th_v, float leak,
                                                   const float* __restrict__ pos,
                                                   int32_t pos_per_member, float* __restrict__ X) {
    typedef float vec __attribute__((ext_vector_type(VEC)));
    const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * VEC;
    const int64_t total = M * d;
    if (e >= total) return;
    const int64_t m = e / ((int64_t)R * d);
    const float* cs[3] = {cq + e, ck + e, cv + e};
    const float ths[3] = {th_q[m], th_k[m], th_v[m]};
    float v[3][VEC], cnt[3][VEC];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int i = 0; i < VEC; ++i) v[q][i] = cnt[q][i] = 0.0f;
#pragma unroll 4
    for (int32_t t = 0; t < T; ++t) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const vec c = *reinterpret_cast<const vec*>(cs[q] + (int64_t)t * total);
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                float s;
                v[q][i] = lif_upd(v[q][i], c[i], leak, ths[q], &s);
                cnt[q][i] = __fadd_rn(cnt[q][i], s);
            }
        }
    }
    const vec p = *reinterpret_cast<const vec*>(pos + (pos_per_member ? e : e - m * R * d));
    vec x;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
        float rate[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) rate[q] = __fdiv_rn(cnt[q][i], (float)T);
        x[i] = __fadd_rn(__fdiv_rn(__fadd_rn(__fadd_rn(rate[0], rate[1]), rate[2]), 3.0f), p[i]);
    }
    *reinterpret_cast<vec*>(X + e) = x;
}

// One head of multihead_attention_once for one member per workgroup
// (snn_self_attention_heads.py:54-70 with row_softmax_lif): Q, K and V of the
// member's R tokens are staged in LDS; each wave takes groups of NQ query rows.
// Per row lane j is key neuron j: h_j = beta (q_i . k_j), normalised by max |h| +
// 1e-6, n_iter LIF steps with the inhibition g_inh * (sum of counts), p_j = count_j /
// (sum count + 1e-6) into the wave's LDS rows; then out_i = p @ V for 64 / hd rows
// at once, lane rr * hd + c summing row rr's channel c over j in index order.
//
// Bound by vector instructions (bits are the reference's, so mul and add stay apart).
// The counts' sum is a scalar: it grows by the population count of the spikes' lane
// mask, so a step needs no reduction over lanes.  Head sizes 8, 16 and 32 have their own
// instances: a lane's key (hd values) and its V column (64) stay in registers over
// its wave's rows, and only the uniform q and the p rows are read from LDS, four at a
// time.  Other sizes read K and V from LDS: no configuration here has them, and an
// instance of 64 would hold 128 values a lane.
// Calls of 1024 members x 4 heads, 64 tokens, 8 steps, against a reduction over lanes in
// every step and K and V from LDS in every group: head size 8 121 -> 71 us, 16 125 -> 85,
// 32 259 -> 107; the general form 4 113 -> 78, 48 660 -> 352, 64 922 -> 503 (17 tokens: 4
// 35 -> 23, 64 147 -> 49).
constexpr int kSaWaves = 4;
constexpr int kSaMaxR = 64, kSaMaxHd = 64;
constexpr int kSaPP = kSaMaxR + 4;  // pitch of a wave's p rows (16-byte reads, distinct banks)
template <int HD, int NQ>
__global__ __launch_bounds__(kSaWaves * 64) void k_sa_attention(
        const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
        int32_t ld, int32_t R, int32_t H, int32_t hd_, const float* __restrict__ beta,
        const float* __restrict__ vth, float g_inh, float leak, int32_t n_iter,
        float* __restrict__ out) {
    extern __shared__ __align__(16) float sa_lds[];
    const int hd = HD ? HD : hd_, pitch = HD ? HD + 4 : hd_ + 1;
    const int m = (int)(blockIdx.x / (uint32_t)H), h = (int)(blockIdx.x % (uint32_t)H);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* ps = sa_lds + w * (NQ * kSaPP);
    float* qs = sa_lds + kSaWaves * NQ * kSaPP;
    float* ks = qs + R * pitch;
    float* vs = ks + R * pitch;
    const int64_t row0 = (int64_t)m * R;
    for (int i = threadIdx.x; i < R * hd; i += kSaWaves * 64) {
        const int r = i / hd, c = i % hd;
        const int64_t g = (row0 + r) * ld + (int64_t)h * hd + c;
        qs[r * pitch + c] = Q[g];
        ks[r * pitch + c] = K[g];
        vs[r * pitch + c] = V[g];
    }
    __syncthreads();
    const float b = beta[m], th = vth[m];
    const bool key = lane < R;
    const uint64_t keys = R == 64 ? ~0ull : (1ull << R) - 1;
    const int rpv = 64 / hd;  // rows of a p @ V pass
    const int rr = lane / hd, cc = lane - rr * hd;
    float kr[HD ? HD : 1], vr[HD ? kSaMaxR : 1];
    if constexpr (HD > 0) {
#pragma unroll
        for (int c = 0; c < HD; ++c) kr[c] = key ? ks[lane * pitch + c] : 0.0f;
#pragma unroll
        for (int j = 0; j < kSaMaxR; ++j) vr[j] = j < R ? vs[j * pitch + cc] : 0.0f;
    }
    for (int i0 = w * NQ; i0 < R; i0 += kSaWaves * NQ) {
        const int nr = min(NQ, R - i0);
        // the group's rows side by side (rows past R repeat row R - 1 and are
        // not stored): independent chains
        float hn[NQ], u[NQ], cnt[NQ];
        int32_t tot[NQ];
        {
            float sd[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) sd[q] = 0.0f;
            if constexpr (HD > 0) {
#pragma unroll
                for (int c = 0; c < HD; c += 4)
#pragma unroll
                    for (int q = 0; q < NQ; ++q) {
                        const float4 x = *reinterpret_cast<const float4*>(
                                qs + min(i0 + q, R - 1) * pitch + c);
                        sd[q] = __fadd_rn(sd[q], __fmul_rn(x.x, kr[c]));
                        sd[q] = __fadd_rn(sd[q], __fmul_rn(x.y, kr[c + 1]));
                        sd[q] = __fadd_rn(sd[q], __fmul_rn(x.z, kr[c + 2]));
                        sd[q] = __fadd_rn(sd[q], __fmul_rn(x.w, kr[c + 3]));
                    }
            } else if (key) {
                for (int c = 0; c < hd; ++c) {
                    const float kv = ks[lane * pitch + c];
#pragma unroll
                    for (int q = 0; q < NQ; ++q)
                        sd[q] = __fadd_rn(sd[q], __fmul_rn(qs[min(i0 + q, R - 1) * pitch + c], kv));
                }
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const float hj = key ? __fmul_rn(b, sd[q]) : 0.0f;
                const float den = __fadd_rn(wmax(key ? fabsf(hj) : 0.0f), 1e-6f);
                hn[q] = __fdiv_rn(hj, den);
                u[q] = 0.0f;
                cnt[q] = 0.0f;
                tot[q] = 0;
            }
        }
        for (int it = 0; it < n_iter; ++it) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const float inh = __fmul_rn(g_inh, (float)tot[q]);
                float sp;
                u[q] = lif_upd(u[q], __fsub_rn(hn[q], inh), leak, th, &sp);
                cnt[q] = __fadd_rn(cnt[q], sp);
                tot[q] += __popcll(__ballot(sp != 0.0f) & keys);
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            if (q < nr) ps[q * kSaPP + lane] = key ? __fdiv_rn(cnt[q], __fadd_rn((float)tot[q], 1e-6f)) : 0.0f;
        // the group's weights are read by other lanes of this wave only
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int q0 = 0; q0 < nr; q0 += rpv) {
            const int q = q0 + rr;
            if (rr < rpv && q < nr) {
                float s = 0.0f;
                const float* pr = ps + q * kSaPP;
                if constexpr (HD > 0) {
#pragma unroll
                    for (int j = 0; j < kSaMaxR; j += 16) {
                        if (j >= R) break;  // past R p and v are 0, and s is never -0
#pragma unroll
                        for (int e = 0; e < 16; e += 4) {
                            const float4 x = *reinterpret_cast<const float4*>(pr + j + e);
                            s = __fadd_rn(s, __fmul_rn(x.x, vr[j + e]));
                            s = __fadd_rn(s, __fmul_rn(x.y, vr[j + e + 1]));
                            s = __fadd_rn(s, __fmul_rn(x.z, vr[j + e + 2]));
                            s = __fadd_rn(s, __fmul_rn(x.w, vr[j + e + 3]));
                        }
                    }
                } else {
                    for (int j = 0; j < R; ++j) s = __fadd_rn(s, __fmul_rn(pr[j], vs[j * pitch + cc]));
                }
                out[(row0 + i0 + q) * ld + (int64_t)h * hd + cc] = s;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// lif_single of ffn_once (snn_self_attention_heads.py:79-83): per row,
// act = c / max(max |c|, 1e-6) >= vth.  One wave per row.
__global__ __launch_bounds__(256) void k_sa_ffn_spike(const float* __restrict__ c, int64_t M,
                                                      int32_t d, int32_t R,
                                                      const float* __restrict__ vth,
                                                      float* __restrict__ act) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= M) return;  // whole wave
    const float* cr = c + row * d;
    float mx = 0.0f;
    for (int32_t j = lane; j < d; j += 64) mx = fmaxf(mx, fabsf(cr[j]));
    const float den = fmaxf(wmax(mx), 1e-6f);
    const float th = vth[row / R];
    for (int32_t j = lane; j < d; j += 64) act[row * d + j] = __fdiv_rn(cr[j], den) >= th ? 1.0f : 0.0f;
}

// x += y (the blocks' residual adds).
__global__ __launch_bounds__(256) void k_add_inplace(float* __restrict__ x,
                                                     const float* __restrict__ y, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) x[e] = __fadd_rn(x[e], y[e]);
}

// jnp.mean(X, axis=0) per member: out[m, c] = (sum_i X[m R + i, c]) / R in
// index order.  One thread per (member, column).
__global__ __launch_bounds__(256) void k_sa_pool(const float* __restrict__ X, int64_t n,
                                                 int32_t R, int32_t d, float* __restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n * d) return;
    const int64_t m = e / d;
    const int32_t c = (int32_t)(e % d);
    float s = 0.0f;
    for (int32_t i = 0; i < R; ++i) s = __fadd_rn(s, X[(m * R + i) * d + c]);
    out[e] = __fdiv_rn(s, (float)R);
}

// y[r, :] *= s[r] (logits * out_gain per member).
__global__ __launch_bounds__(256) void k_scale_rows(float* __restrict__ y, int64_t rows,
                                                    int32_t cols, const float* __restrict__ s) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < rows * cols) y[e] = __fmul_rn(y[e], s[e / cols]);
}

static uint32_t blocks256(int64_t n) { return (uint32_t)((n + 255) / 256); }

}  // namespace hses

using namespace hses;

extern "C" int hses_softplus(const float* d_x, int64_t n, float* d_y, void* stream) {
    HSES_REQUIRE(n >= 0, "negative length");
    if (n == 0) return HSES_OK;
    HSES_REQUIRE(d_x && d_y, "NULL pointer");
    HSES_REQUIRE((n + 255) / 256 < (1ll << 31), "grid too large");
    hipLaunchKernelGGL(k_softplus, dim3(blocks256(n)), dim3(256), 0, (hipStream_t)stream, d_x, n, d_y);
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

extern "C" int hses_sa_encode(const float* d_cq, const float* d_ck, const float* d_cv, int32_t T,
                              int64_t M, int32_t d, int32_t rows_per_member, const float* d_th_q,
                              const float* d_th_k, const float* d_th_v, float tau_m,
                              const float* d_pos, int32_t pos_per_member, float* d_X,
                              void* stream) {
    HSES_REQUIRE(T >= 1 && M >= 0 && d >= 1 && rows_per_member >= 1, "bad sizes");
    HSES_REQUIRE(M % rows_per_member == 0, "rows are not a whole number of members");
    HSES_REQUIRE(tau_m > 0.0f, "tau_m must be > 0");
    if (M == 0) return HSES_OK;
    HSES_REQUIRE(d_cq && d_ck && d_cv && d_th_q && d_th_k && d_th_v && d_pos && d_X, "NULL pointer");
    HSES_REQUIRE(d_X != d_cq && d_X != d_ck && d_X != d_cv, "X must not alias the currents");
    HSES_REQUIRE((M * d + 255) / 256 < (1ll << 31), "grid too large");
    const uintptr_t bases = reinterpret_cast<uintptr_t>(d_cq) | reinterpret_cast<uintptr_t>(d_ck) |
                            reinterpret_cast<uintptr_t>(d_cv) | reinterpret_cast<uintptr_t>(d_pos) |
                            reinterpret_cast<uintptr_t>(d_X);
    const bool vec = d % 4 == 0 && bases % 16 == 0;
    auto launch = [&](auto kernel, int64_t threads) {
        hipLaunchKernelGGL(kernel, dim3(blocks256(threads)), dim3(256), 0, (hipStream_t)stream, d_cq,
                           d_ck, d_cv, T, M, d, rows_per_member, d_th_q, d_th_k, d_th_v, 1.0f / tau_m,
                           d_pos, pos_per_member, d_X);
    };
    if (vec)
        launch(k_sa_encode<4>, M * d / 4);
    else
        launch(k_sa_encode<1>, M * d);
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

extern "C" int hses_sa_attention(const float* d_q, const float* d_k, const float* d_v,
                                 int32_t ld, int64_t n, int32_t R, int32_t H, int32_t hd,
                                 const float* d_beta, const float* d_vth, float g_inh, float tau_m,
                                 int32_t n_iter, float* d_out, void* stream) {
    HSES_REQUIRE(n >= 0 && H >= 1 && n_iter >= 0, "bad sizes");
    HSES_REQUIRE(R >= 1 && R <= kSaMaxR, "tokens per member must be in [1, 64]");
    HSES_REQUIRE(hd >= 1 && hd <= kSaMaxHd, "head size must be in [1, 64]");
    HSES_REQUIRE(ld >= H * hd, "row stride smaller than the heads");
    HSES_REQUIRE(tau_m > 0.0f, "tau_m must be > 0");
    if (n == 0) return HSES_OK;
    HSES_REQUIRE(d_q && d_k && d_v && d_beta && d_vth && d_out, "NULL pointer");
    HSES_REQUIRE(d_out != d_q && d_out != d_k && d_out != d_v, "out must not alias q, k or v");
    HSES_REQUIRE(n * H < (1ll << 31), "grid too large");
    auto launch = [&](auto kernel, int nq, int pitch) {
        const size_t lds = ((size_t)kSaWaves * nq * kSaPP + 3 * (size_t)R * pitch) * sizeof(float);
        hipLaunchKernelGGL(kernel, dim3((uint32_t)(n * H)), dim3(kSaWaves * 64), lds, (hipStream_t)stream,
                           d_q, d_k, d_v, ld, R, H, hd, d_beta, d_vth, g_inh, 1.0f / tau_m, n_iter, d_out);
    };
    switch (hd) {  // 8: eight rows fill a p @ V pass
        case 8: launch(k_sa_attention<8, 8>, 8, hd + 4); break;
        case 16: launch(k_sa_attention<16, 4>, 4, hd + 4); break;
        case 32: launch(k_sa_attention<32, 4>, 4, hd + 4); break;
        default: launch(k_sa_attention<0, 4>, 4, hd + 1); break;
    }
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

extern "C" int hses_sa_ffn_spike(const float* d_c, int64_t M, int32_t d, int32_t rows_per_member,
                                 const float* d_vth, float* d_act, void* stream) {
    HSES_REQUIRE(M >= 0 && d >= 1 && rows_per_member >= 1, "bad sizes");
    HSES_REQUIRE(M % rows_per_member == 0, "rows are not a whole number of members");
    if (M == 0) return HSES_OK;
    HSES_REQUIRE(d_c && d_vth && d_act, "NULL pointer");
    HSES_REQUIRE((M + 3) / 4 < (1ll << 31), "grid too large");
    hipLaunchKernelGGL(k_sa_ffn_spike, dim3((uint32_t)((M + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, d_c, M, d, rows_per_member, d_vth, d_act);
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

extern "C" int hses_add_inplace(float* d_x, const float* d_y, int64_t n, void* stream) {
    HSES_REQUIRE(n >= 0, "negative length");
    if (n == 0) return HSES_OK;
    HSES_REQUIRE(d_x && d_y, "NULL pointer");
    HSES_REQUIRE((n + 255) / 256 < (1ll << 31), "grid too large");
    hipLaunchKernelGGL(k_add_inplace, dim3(blocks256(n)), dim3(256), 0, (hipStream_t)stream, d_x,
                       d_y, n);
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

extern "C" int hses_sa_pool(const float* d_X, int64_t n, int32_t R, int32_t d, float* d_out,
                            void* stream) {
    HSES_REQUIRE(n >= 0 && R >= 1 && d >= 1, "bad sizes");
    if (n == 0) return HSES_OK;
    HSES_REQUIRE(d_X && d_out, "NULL pointer");
    HSES_REQUIRE((n * d + 255) / 256 < (1ll << 31), "grid too large");
    hipLaunchKernelGGL(k_sa_pool, dim3(blocks256(n * d)), dim3(256), 0, (hipStream_t)stream, d_X,
                       n, R, d, d_out);
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

extern "C" int hses_scale_rows(float* d_y, int64_t rows, int32_t cols, const float* d_s,
                               void* stream) {
    HSES_REQUIRE(rows >= 0 && cols >= 1, "bad sizes");
    if (rows == 0) return HSES_OK;
    HSES_REQUIRE(d_y && d_s, "NULL pointer");
    HSES_REQUIRE((rows * cols + 255) / 256 < (1ll << 31), "grid too large");
    hipLaunchKernelGGL(k_scale_rows, dim3(blocks256(rows * cols)), dim3(256), 0,
                       (hipStream_t)stream, d_y, rows, cols, d_s);
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}
