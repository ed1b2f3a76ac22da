// linear_bf16.hip -- bf16 perturbed forward for outputs at least 256 wide at
// ranks up to 4:
//   do_mm  (eggroll.rs:419-446):  y = x W^T + (x B_m) A_m^T,
//   do_Tmm (eggroll.rs:450-477):  y = x W + (x A_m) B_m^T,
// with an optional elementwise activation and an fp32 or bf16 output (the
// Linear / Tmm layers of the RWKV-7 LM, llm.rs:182-480).
//
// W is converted once per call to bf16 (output rows x kp, transposed for
// do_Tmm) and k_factors draws every member's factor rows; then
//   k_gemm_bf16_dl (rank 0 or 1, K a multiple of 32): 128 x 256 tiles fed by
//   direct-to-LDS loads, the rank-1 terms on the matrix cores too (below);
//   k_gemm_bf16 (the rest): a 256 x 256 output tile per workgroup; 8 waves of 64
//   rows x 128 columns on bf16 MFMA 32x32x16 with fp32 accumulation.  K runs in
//   steps of 64, double-buffered in LDS: right after a step's barrier every thread
//   issues the next step's x and W loads into registers, the waves run the
//   step's MFMAs, and the registers go to the other buffer before the next
//   barrier.  Each thread also accumulates x B_m for its row and 32-column
//   half of the step on the vector ALU (x as staged, the input-side factor
//   rounded to bf16, fp32 sums); the epilogue adds (x B_m) A_m^T with the
//   output-side factor in fp32, applies the activation and stores.
// Tiles are ordered so that each XCD (workgroups are dealt to the 8 in turn)
// works through a contiguous range with the column tiles of a row tile
// adjacent: the workgroups reading one x row tile share an L2.
#include <math.h>

#include <type_traits>

#include "linear_common.h"
#include "mfma.h"
#include "runtime.h"

namespace hses {

constexpr int KB_BM = 256, KB_BN = 256, KB_BK = 64, KB_THREADS = 512;
constexpr int KB_P = KB_BK + 8;        // LDS pitch of an x / W row (bf16): 144 B
constexpr int KB_BUF = KB_BM * KB_P;   // bf16 elements of one x (or W) buffer
constexpr int KB_RMAX = 4;
constexpr int KB_BPT = 2;              // input-side factor values staged per thread and step

// The direct-to-LDS kernel k_gemm_bf16_dl (rank 0 or 1, K a multiple of 32): a 128 x 256 tile and four waves, K steps of 32 in three LDS stages, two
// steps' loads in flight during a step.  A stage holds x and W rows of 64 bytes,
// 16-byte piece c of row r in slot c ^ ((r / 4) % 4), so one
// global_load_lds_dwordx4 fills 16 rows (lane p: row p / 4, slot p % 4) and the
// MFMA operand reads of eight lanes (eight rows, one piece) hit distinct banks;
// then the members' input-side factors of the step (bf16, one more load).  fp32 x
// goes through registers, rounded to bf16, into the same places.
constexpr int DL_BM = 128, DL_BK = 32, DL_NS = 3, DL_THREADS = 256;
constexpr int DL_NM = 4;                          // members a tile may touch
constexpr int DL_XB = DL_BM * DL_BK * 2;          // bytes of x per stage
constexpr int DL_WB = KB_BN * DL_BK * 2;          // bytes of W per stage
constexpr int DL_FB = DL_NM * DL_BK * 2;          // bytes of factor values per stage
constexpr int DL_SB = DL_XB + DL_WB + DL_FB;      // 24832 bytes per stage

typedef float f32x16b __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2b __attribute__((ext_vector_type(2)));

// a.lo b.lo + a.hi b.hi + c for bf16 pairs (v_dot2c_f32_bf16)
__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2b, a), __builtin_bit_cast(bf16x2b, b),
                                           c, false);
}

__device__ __forceinline__ f32x16b mfma32b(const u16x8& a, const u16x8& b, f32x16b c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int ACT>
__device__ __forceinline__ float act_value(float v) {
    if constexpr (ACT == ACT_TANH) return tanhf(v);
    if constexpr (ACT == ACT_SIGMOID) return 1.0f / (1.0f + expf(-v));
    if constexpr (ACT == ACT_RELU_SQ) {
        const float z = v > 0.0f ? v : 0.0f;
        return z * z;
    }
    return v;
}

// s_waitcnt vmcnt(N) (expcnt and lgkmcnt not waited for), gfx9 encoding
template <int N>
__device__ __forceinline__ void vm_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// RK: rank padded to 1 or 4 (zeros past r).  bch: words of one step's staged
// input-side factor rows, as bf16 pairs of consecutive k ([lm][32][RK], 0
// without noise).  x and W go through registers, one 64-wide step ahead.
template <int XFMT, int RK>
__global__ __launch_bounds__(KB_THREADS)
void k_gemm_bf16(LinParams P, const uint16_t* __restrict__ Wb, int32_t kp, const float* __restrict__ F,
                 int32_t bch, int32_t act, int32_t ybf16, int32_t vec_y) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint16_t* Xs = reinterpret_cast<uint16_t*>(smem);   // [2][256][KB_P]
    uint16_t* Ws = Xs + 2 * KB_BUF;                      // [2][256][KB_P]
    uint32_t* Bc = reinterpret_cast<uint32_t*>(Ws + 2 * KB_BUF);  // [2][bch] bf16 pairs
    float* As = reinterpret_cast<float*>(Bc + 2 * bch);           // [lm][256][RK]

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lc = lane & 31, hl = lane >> 5;
    const int wr = wave >> 1, wc = wave & 1;  // wave tile: rows 64 wr.., columns 128 wc..
    int64_t L0;
    int32_t o0;
    {
        const uint32_t nb = gridDim.x, g = blockIdx.x, xcd = g & 7u, j = g >> 3;
        const uint32_t q = nb >> 3, rem = nb & 7u;
        const uint32_t ncol = (uint32_t)((P.a + KB_BN - 1) / KB_BN);
        const uint32_t t = ncol == 1 ? g
                           : xcd < rem ? xcd * (q + 1) + j : rem * (q + 1) + (xcd - rem) * q + j;
        L0 = (int64_t)(t / ncol) * KB_BM;
        o0 = (int32_t)(t % ncol) * KB_BN;
    }
    const int32_t a = P.a, b = P.b, r = P.r;
    const int32_t rows_here = (int32_t)min<int64_t>(KB_BM, P.total - L0);
    const TileRows tr(P, L0);
    const int32_t nm = tr.member(P, rows_here - 1) + 1;
    const bool noisy = r > 0;
    const int64_t fpitch = (int64_t)(a + b) * r;
    const float* Fm = F + (int64_t)tr.m_first * fpitch;
    const int32_t in_off = P.tmm ? a : 0, out_off = P.tmm ? 0 : b;  // factor rows by role

    // ---- output-side factor rows of the tile's columns (fp32) ------------------
    if (noisy) {
        for (int32_t i = tid; i < nm * KB_BN * RK; i += KB_THREADS) {
            const int32_t c = i % RK, o = (i / RK) % KB_BN, lm = i / (RK * KB_BN);
            As[i] = (c < r && o0 + o < a) ? Fm[lm * fpitch + (int64_t)(out_off + o0 + o) * r + c]
                                          : 0.0f;
        }
    }

    // ---- staging and the K loop ---------------------------------------------------
    f32x16b acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    // x B_m from the MFMA x operands: the two waves that share rows 64 wr ..
    // take one 32-row block each (block wc), so every SIMD does the same share;
    // lane (lc, hl) holds k 16 ks + 8 hl .. + 8 of row xbr
    const int32_t xbr = wr * 64 + 32 * wc + lc;
    const int32_t xbm = xbr < rows_here ? tr.member(P, xbr) : 0;  // its member in the tile
    float xb[RK];
#pragma unroll
    for (int c = 0; c < RK; ++c) xb[c] = 0.0f;

    // ---- staging: thread -> x row tid / 2 and W row tid / 2, 32 k each ----------
    const int xr = tid >> 1, xk = (tid & 1) * 32;
    const bool xvalid = xr < rows_here;
    const int64_t xoff = xvalid ? tr.offset(P, xr, P.x_stride, P.x_plane) : 0;
    const int32_t wrow = o0 + xr;
    const bool wvalid = wrow < a;
    const uint16_t* wsrc = Wb + (int64_t)(wvalid ? wrow : 0) * kp + xk;
    constexpr int XU = XFMT == HSES_FMT_F32 ? 8 : 4;  // 16-byte loads of x per thread and step
    constexpr int XE = XFMT == HSES_FMT_F32 ? 4 : 8;  // elements per 16-byte load
    uint4 xv[XU], wv[4];
    uint32_t bv[KB_BPT];
    // staged factor words of this thread: (member, k pair, rank column), the
    // source of the pair's first k at step 0 (a step adds 64 rows)
    const float* bsrc[KB_BPT];
    int32_t bk2[KB_BPT];
    bool bon[KB_BPT];
#pragma unroll
    for (int j = 0; j < KB_BPT; ++j) {
        const int32_t e = tid + KB_THREADS * j;  // [lm][kp][c]
        const int32_t c = e % RK, kp2 = (e / RK) % (KB_BK / 2), lm = e / (RK * (KB_BK / 2));
        bon[j] = noisy && e < bch && lm < nm && c < r;
        bk2[j] = 2 * kp2;
        bsrc[j] = Fm + (bon[j] ? lm * fpitch + (int64_t)(in_off + 2 * kp2) * r + c : 0);
    }
    auto load_step = [&](int32_t kt) {
        const int32_t k0 = kt * KB_BK + xk;
        // whole steps load unconditionally; the last, partial one masks
        if (xvalid && k0 + 32 <= b) {
#pragma unroll
            for (int q = 0; q < XU; ++q) {
                if constexpr (XFMT == HSES_FMT_F32)
                    xv[q] = reinterpret_cast<const uint4*>(static_cast<const float*>(P.x) + xoff + k0)[q];
                else
                    xv[q] = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(P.x) + xoff + k0)[q];
            }
        } else {
#pragma unroll
            for (int q = 0; q < XU; ++q) {
                const bool ok = xvalid && k0 + XE * q < b;
                if constexpr (XFMT == HSES_FMT_F32)
                    xv[q] = ok ? reinterpret_cast<const uint4*>(static_cast<const float*>(P.x) + xoff + k0)[q]
                               : uint4{0, 0, 0, 0};
                else
                    xv[q] = ok ? reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(P.x) + xoff + k0)[q]
                               : uint4{0, 0, 0, 0};
            }
        }
        if (wvalid) {
#pragma unroll
            for (int q = 0; q < 4; ++q) wv[q] = reinterpret_cast<const uint4*>(wsrc + kt * KB_BK)[q];
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) wv[q] = uint4{0, 0, 0, 0};
        }
        if (noisy) {
#pragma unroll
            for (int j = 0; j < KB_BPT; ++j) {
                const bool ok = bon[j] && kt * KB_BK + bk2[j] < b;  // b is even: both k of the pair
                const float* p = bsrc[j] + (int64_t)kt * KB_BK * r;
                bv[j] = ok ? pack_bf16x2(p[0], p[r]) : 0u;
            }
        }
    };
    auto store_step = [&](int buf) {
        uint16_t* xd = Xs + buf * KB_BUF + xr * KB_P + xk;
        if constexpr (XFMT == HSES_FMT_F32) {
#pragma unroll
            for (int q = 0; q < XU; q += 2) {
                const uint4 lo = xv[q], hi = xv[q + 1];
                *reinterpret_cast<uint4*>(xd + 4 * q) = uint4{
                    pack_bf16x2(__uint_as_float(lo.x), __uint_as_float(lo.y)),
                    pack_bf16x2(__uint_as_float(lo.z), __uint_as_float(lo.w)),
                    pack_bf16x2(__uint_as_float(hi.x), __uint_as_float(hi.y)),
                    pack_bf16x2(__uint_as_float(hi.z), __uint_as_float(hi.w))};
            }
        } else {
#pragma unroll
            for (int q = 0; q < XU; ++q) *reinterpret_cast<uint4*>(xd + 8 * q) = xv[q];
        }
        uint16_t* wd = Ws + buf * KB_BUF + xr * KB_P + xk;
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<uint4*>(wd + 8 * q) = wv[q];
        if (noisy) {
#pragma unroll
            for (int j = 0; j < KB_BPT; ++j) {
                const int32_t e = tid + KB_THREADS * j;
                if (e < bch) Bc[buf * bch + e] = bv[j];
            }
        }
    };

    const int32_t nkt = (b + KB_BK - 1) / KB_BK;
    load_step(0);
    store_step(0);
    __syncthreads();
    for (int32_t kt = 0; kt < nkt; ++kt) {
        const int cur = kt & 1;
        if (kt + 1 < nkt) load_step(kt + 1);
        const uint16_t* X = Xs + cur * KB_BUF;
        const uint16_t* W = Ws + cur * KB_BUF;
#pragma unroll
        for (int ks = 0; ks < KB_BK / 16; ++ks) {
            const int kk = ks * 16 + hl * 8;
            u16x8 af[2], bf[4];
#pragma unroll
            for (int i = 0; i < 2; ++i) af[i] = lds_u16x8(X + (wr * 64 + 32 * i + lc) * KB_P + kk);
#pragma unroll
            for (int j = 0; j < 4; ++j) bf[j] = lds_u16x8(W + (wc * 128 + 32 * j + lc) * KB_P + kk);
            // D = W x^T: a lane's accumulator holds one output row (its x row)
            // and runs of four consecutive output columns
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mfma32b(bf[j], af[i], acc[i][j]);
            if (noisy) {
                // the factor's bf16 pairs of these 8 k: [lm][pair][c]
                const uint4* bs = reinterpret_cast<const uint4*>(
                    Bc + cur * bch + (xbm * (KB_BK / 2) + ks * 8 + hl * 4) * RK);
                const uint4 xw = __builtin_bit_cast(uint4, wc ? af[1] : af[0]);
                const uint32_t xp[4] = {xw.x, xw.y, xw.z, xw.w};
                if constexpr (RK == 1) {
                    const uint4 q = bs[0];  // pairs u = 0..3
                    xb[0] = dot2_bf16(xp[0], q.x, xb[0]);
                    xb[0] = dot2_bf16(xp[1], q.y, xb[0]);
                    xb[0] = dot2_bf16(xp[2], q.z, xb[0]);
                    xb[0] = dot2_bf16(xp[3], q.w, xb[0]);
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const uint4 q = bs[u];  // rank columns 0..3 of pair u
                        xb[0] = dot2_bf16(xp[u], q.x, xb[0]);
                        xb[1] = dot2_bf16(xp[u], q.y, xb[1]);
                        xb[2] = dot2_bf16(xp[u], q.z, xb[2]);
                        xb[3] = dot2_bf16(xp[u], q.w, xb[3]);
                    }
                }
            }
        }
        if (kt + 1 < nkt) store_step(cur ^ 1);
        __syncthreads();
    }

    // ---- epilogue: y = act(x W^T + (x B_m) A_m^T) ---------------------------------
    float* XBs = reinterpret_cast<float*>(Xs);  // [256][RK]; the buffers are free now
    if (noisy) {
#pragma unroll
        for (int c = 0; c < RK; ++c) {
            const float v = xb[c] + __shfl_xor(xb[c], 32);  // the two k groups
            if (hl == 0) XBs[xbr * RK + c] = v;
        }
        __syncthreads();
    }
    // One copy of the store loop per (activation, output format), chosen once.
    // With D = W x^T, accumulator element e of lane l is output row lc of the
    // 32-row block and column 8 (e / 4) + 4 hl + e % 4 of the 32-column tile:
    // each lane owns two rows and stores four consecutive columns at a time.
    const bool flat = P.n_time == 1;
    auto store_all = [&](auto actc, auto ybc) __attribute__((always_inline)) {
        constexpr int ACT = decltype(actc)::value;
        constexpr bool YB = decltype(ybc)::value;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int32_t row = wr * 64 + 32 * i + lc;
            if (row >= rows_here) continue;
            const int32_t lm = noisy ? tr.member(P, row) : 0;
            const int64_t yoff =
                (flat ? (L0 + row) * P.y_stride : tr.offset(P, row, P.y_stride, P.y_plane)) + o0;
            float xr_[RK];
#pragma unroll
            for (int c = 0; c < RK; ++c) xr_[c] = noisy ? XBs[row * RK + c] : 0.0f;
            if constexpr (YB) {
                if (vec_y == 2 && o0 + KB_BN <= a) {
                    // lanes l and l + 32 hold columns 8 g + 0..3 and 8 g + 4..7: after a
                    // swap of the upper half-lanes of group g with the lower of group
                    // g + 1, lane l holds the 8 columns of group g and lane l + 32 those
                    // of g + 1: one 16-byte store each
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int g = 0; g < 4; g += 2) {
                            uint32_t w[2][2];
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                const int32_t c0 = wc * 128 + 32 * j + 8 * (g + h) + 4 * hl;
                                float v[4];
#pragma unroll
                                for (int u = 0; u < 4; ++u) v[u] = acc[i][j][4 * (g + h) + u];
                                if (noisy) {
                                    const float* ar = As + ((size_t)lm * KB_BN + c0) * RK;
#pragma unroll
                                    for (int u = 0; u < 4; ++u) {
                                        float z = 0.0f;
#pragma unroll
                                        for (int c = 0; c < RK; ++c)
                                            z = __fadd_rn(z, __fmul_rn(xr_[c], ar[u * RK + c]));
                                        v[u] = __fadd_rn(v[u], z);
                                    }
                                }
#pragma unroll
                                for (int u = 0; u < 4; ++u) v[u] = act_value<ACT>(v[u]);
                                w[h][0] = pack_bf16x2(v[0], v[1]);
                                w[h][1] = pack_bf16x2(v[2], v[3]);
                            }
#pragma unroll
                            for (int q = 0; q < 2; ++q) {
                                const auto sw = __builtin_amdgcn_permlane32_swap(w[0][q], w[1][q], false, false);
                                w[0][q] = sw[0];
                                w[1][q] = sw[1];
                            }
                            const int32_t cs = wc * 128 + 32 * j + 8 * (g + hl);
                            *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(P.y) + yoff + cs) =
                                uint4{w[0][0], w[0][1], w[1][0], w[1][1]};
                        }
                    continue;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int32_t col0 = wc * 128 + 32 * j + 8 * g + 4 * hl;
                    float v[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = acc[i][j][4 * g + u];
                    if (noisy) {
                        const float* ar = As + ((size_t)lm * KB_BN + col0) * RK;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            float z = 0.0f;
#pragma unroll
                            for (int c = 0; c < RK; ++c) z = __fadd_rn(z, __fmul_rn(xr_[c], ar[u * RK + c]));
                            v[u] = __fadd_rn(v[u], z);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = act_value<ACT>(v[u]);
                    if (vec_y && o0 + col0 + 4 <= a) {
                        if constexpr (YB)
                            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(P.y) + yoff + col0) =
                                uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                        else
                            *reinterpret_cast<float4*>(P.y + yoff + col0) = float4{v[0], v[1], v[2], v[3]};
                    } else {
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            if (o0 + col0 + u >= a) continue;
                            if constexpr (YB)
                                reinterpret_cast<uint16_t*>(P.y)[yoff + col0 + u] = f2bf(v[u]);
                            else
                                P.y[yoff + col0 + u] = v[u];
                        }
                    }
                }
        }
    };
    using T0 = std::integral_constant<int, ACT_NONE>;
    using T1 = std::integral_constant<int, ACT_TANH>;
    using T2 = std::integral_constant<int, ACT_SIGMOID>;
    using T3 = std::integral_constant<int, ACT_RELU_SQ>;
    auto by_act = [&](auto ybc) __attribute__((always_inline)) {
        switch (act) {
            case ACT_TANH: store_all(T1{}, ybc); break;
            case ACT_SIGMOID: store_all(T2{}, ybc); break;
            case ACT_RELU_SQ: store_all(T3{}, ybc); break;
            default: store_all(T0{}, ybc); break;
        }
    };
    if (ybf16) by_act(std::true_type{});
    else by_act(std::false_type{});
}

// Whether the three bf16 parts of a rank-1 operand hold all of it (zero, or a size
// whose last part and part products stay in the normal ranges; not NaN).
__device__ __forceinline__ bool parts_whole(float v) {
    const float a = fabsf(v);
    return a == 0.0f || (a >= 0x1p-50f && a <= 0x1p60f);
}

// The same product at rank 0 or 1 (see DL_BM).  x B_m and the rank-1 term are
// matrix products, so the matrix cores form them (on the vector ALU they were
// 2900 instructions per wave and tile, more issue time than the MFMAs):
//   x B_m   a ninth MFMA per k slice: the tile's members' factor rows are a fifth
//           column tile (one lane column per member, at most DL_NM), formed once
//           per 32-row block (wave column wc takes block wc of its rows);
//   (x B_m) A_m^T   one k slice at the end.  Each fp32 factor is the sum of three
//           bf16 parts (8 significant bits each), and the six products p + q <= 2
//           fill 6 of the 8 k of a lane: half a slice per member, so the term keeps
//           fp32 accuracy and one rounding.  An output with a factor or an x B_m
//           outside 2^-50 .. 2^60 (parts_whole) takes their fp32 product instead.
// F: the output-side factor rows (fp32, member pitch a + b); Fb: the input-side
// rows as bf16 (member pitch b).
// At 100000 x 512 -> 2048 (bf16 x and y, relu^2, 100 rows per member) the call
// went from 357 to 337 us with the swizzle on r / 4 (LDS conflict cycles 21 M ->
// 4.8 M; 16 lanes of a 16-byte read are served together over 64 banks), the matrix
// terms and the row-wise stores; 32 -> 512 with fp32 y 127 -> 109 us.  It is bound
// by its K loop (293 us without stores): LDS reads (14 KB per wave and step) and
// MFMAs (1152 cycles per step and SIMD) overlap by half.
template <int XFMT, bool NOISY>
__global__ __launch_bounds__(DL_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_bf16_dl(LinParams P, const uint16_t* __restrict__ Wb, int32_t kp, const float* __restrict__ F,
                    const uint16_t* __restrict__ Fb, int32_t act, int32_t ybf16, int32_t vec_y) {
    constexpr bool XF = XFMT == HSES_FMT_F32;
    extern __shared__ __align__(16) unsigned char smem[];  // [DL_NS][DL_SB]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lc = lane & 31, hl = lane >> 5;
    const int wr = wave >> 1;                                      // wave tile: rows 64 wr ..
    const int wc = __builtin_amdgcn_readfirstlane(wave & 1);       // .. columns 128 wc ..
    int64_t L0;
    int32_t o0;
    {
        const uint32_t nb = gridDim.x, g = blockIdx.x, xcd = g & 7u, j = g >> 3;
        const uint32_t q = nb >> 3, rem = nb & 7u;
        const uint32_t ncol = (uint32_t)((P.a + KB_BN - 1) / KB_BN);
        const uint32_t t = ncol == 1 ? g
                           : xcd < rem ? xcd * (q + 1) + j : rem * (q + 1) + (xcd - rem) * q + j;
        L0 = (int64_t)(t / ncol) * DL_BM;
        o0 = (int32_t)(t % ncol) * KB_BN;
    }
    const int32_t a = P.a, b = P.b;
    const int32_t rows_here = (int32_t)min<int64_t>(DL_BM, P.total - L0);
    const TileRows tr(P, L0);
    const int32_t nm = tr.member(P, rows_here - 1) + 1;
    const bool flat = P.n_time == 1;
    auto row_off = [&](int32_t i, int64_t stride, int64_t plane) {
        return flat ? (L0 + i) * stride : tr.offset(P, i, stride, plane);
    };

    // the output-side factors of this thread's column, for the epilogue
    float ao[DL_NM];
    if constexpr (NOISY) {
        const float* f = F + (int64_t)tr.m_first * (a + b) + (P.tmm ? 0 : b) + min(o0 + tid, a - 1);
#pragma unroll
        for (int m = 0; m < DL_NM; ++m) ao[m] = m < nm ? f[(int64_t)m * (a + b)] : 0.0f;
    }

    f32x16b acc[2][4], xba;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        xba[e] = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j][e] = 0.0f;
    }

    const int dr = lane >> 2, dc = (lane & 3) ^ ((lane >> 4) & 3);  // row of 16, k piece
    const uint16_t* xsrc[2];
    const uint16_t* wsrc[4];
    // wave w fills rows 32w .. of x and 64w .. of W, 16 at a time; rows past the
    // tile read row 0 (finite values in rows and columns that are never stored)
    // (fp32 x: thread t loads 16 k of row t / 2)
    const float* xfsrc = nullptr;
    if constexpr (XF) {
        const int32_t R = tid >> 1;
        xfsrc = static_cast<const float*>(P.x) +
                row_off(R < rows_here ? R : 0, P.x_stride, P.x_plane) + (tid & 1) * 16;
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int32_t R = 32 * wave + 16 * h + dr;
            xsrc[h] = static_cast<const uint16_t*>(P.x) +
                      row_off(R < rows_here ? R : 0, P.x_stride, P.x_plane) + dc * 8;
        }
    }
    f32x4 xv[4];
    auto load_x = [&](int32_t st) {
#pragma unroll
        for (int q = 0; q < 4; ++q) xv[q] = reinterpret_cast<const f32x4*>(xfsrc + st * DL_BK)[q];
    };
    auto store_x = [&](int32_t slot) {
        const int R = tid >> 1;
        unsigned char* d = smem + slot * DL_SB + R * 64;
#pragma unroll
        for (int q = 0; q < 2; ++q)
            *reinterpret_cast<uint4*>(d + (((2 * (tid & 1) + q) ^ ((R >> 2) & 3)) << 4)) =
                uint4{pack_bf16x2(xv[2 * q][0], xv[2 * q][1]), pack_bf16x2(xv[2 * q][2], xv[2 * q][3]),
                      pack_bf16x2(xv[2 * q + 1][0], xv[2 * q + 1][1]),
                      pack_bf16x2(xv[2 * q + 1][2], xv[2 * q + 1][3])};
    };
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int32_t R = 64 * wave + 16 * h + dr;
        wsrc[h] = Wb + (int64_t)(o0 + R < a ? o0 + R : 0) * kp + dc * 8;
    }
    // factor rows: lane p holds member p / 4, k piece p % 4 of the step (every
    // wave loads them: the same bytes)
    const bool f_on = NOISY && lane < nm * 4;
    const uint16_t* fsrc = Fb + (f_on ? (int64_t)(tr.m_first + (lane >> 2)) * b + (lane & 3) * 8 : 0);
    auto issue = [&](int32_t st, int32_t slot) {
        unsigned char* base = smem + slot * DL_SB;
        if constexpr (!XF) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                __builtin_amdgcn_global_load_lds(xsrc[h] + st * DL_BK, base + (2 * wave + h) * 1024, 16, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < 4; ++h)
            __builtin_amdgcn_global_load_lds(wsrc[h] + st * DL_BK, base + DL_XB + (4 * wave + h) * 1024,
                                             16, 0, 0);
        if (f_on)
            __builtin_amdgcn_global_load_lds(fsrc + st * DL_BK, base + DL_XB + DL_WB, 16, 0, 0);
    };
    const int32_t nkt = b / DL_BK;
    // The factor loads into registers above are older than every stage load, so
    // the counted waits below cover them too.
    if constexpr (XF) {
        load_x(0);
        store_x(0);
        if (nkt > 1) {
            load_x(1);
            store_x(1);
        }
    }
    issue(0, 0);
    if (nkt > 1) issue(1, 1);
    // operand byte offsets of the rows; the slot depends on the slice
    int32_t aoff[2], boff[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) aoff[i] = (64 * wr + 32 * i + lc) * 64;
#pragma unroll
    for (int j = 0; j < 4; ++j) boff[j] = DL_XB + (128 * wc + 32 * j + lc) * 64;
    const int32_t foff = DL_XB + DL_WB + min(lc, nm - 1) * 64 + hl * 16;
    int32_t slot = 0;
    for (int32_t kt = 0; kt < nkt; ++kt) {
        // this wave's loads of stage kt are done; those of kt + 1 (six, or four
        // with fp32 x, and the factors') stay in flight
        constexpr int NL = XF ? 4 : 6;
        if (kt + 1 == nkt) vm_wait<0>();
        else vm_wait<NL + NOISY>();
        if constexpr (XF) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // store_x
        // every wave's loads of stage kt are in LDS, and every wave is done with
        // stage kt - 1, whose buffer the load of stage kt + 2 reuses
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);  // nothing of this step moves above the wait
        const int32_t slot2 = slot == 0 ? 2 : slot - 1;  // stage kt + 2
        if (kt + 2 < nkt) {
            if constexpr (XF) load_x(kt + 2);  // older than the stage's other loads
            issue(kt + 2, slot2);
        }
        const unsigned char* base = smem + slot * DL_SB;
        slot = slot == 2 ? 0 : slot + 1;
        u16x8 fa[2][2], fb[2][4], ff[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int32_t cx = ((2 * ks + hl) ^ ((lc >> 2) & 3)) << 4;  // this lane's k piece
#pragma unroll
            for (int i = 0; i < 2; ++i) fa[ks][i] = *reinterpret_cast<const u16x8*>(base + aoff[i] + cx);
#pragma unroll
            for (int j = 0; j < 4; ++j) fb[ks][j] = *reinterpret_cast<const u16x8*>(base + boff[j] + cx);
            if constexpr (NOISY) ff[ks] = *reinterpret_cast<const u16x8*>(base + foff + 32 * ks);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mfma32b(fb[ks][j], fa[ks][i], acc[i][j]);
            if constexpr (NOISY) {
                const uint4 x0 = __builtin_bit_cast(uint4, fa[ks][0]), x1 = __builtin_bit_cast(uint4, fa[ks][1]);
                const uint4 xw = uint4{wc ? x1.x : x0.x, wc ? x1.y : x0.y, wc ? x1.z : x0.z, wc ? x1.w : x0.w};
                xba = mfma32b(ff[ks], __builtin_bit_cast(u16x8, xw), xba);
            }
        }
        if constexpr (XF)
            if (kt + 2 < nkt) store_x(slot2);
    }

    // ---- (x B_m) A_m^T as one k slice per two members --------------------------------
    if constexpr (NOISY) {
        __syncthreads();  // every wave is past its last read of the stages
        uint4* AF = reinterpret_cast<uint4*>(smem);  // [nm][256] output-side fragments
        uint4* XF = AF + DL_NM * KB_BN;              // [128] x B_m fragments
        float* AO = reinterpret_cast<float*>(XF + DL_BM);  // the operands themselves
        float* XB = AO + DL_NM * KB_BN;
        // products k: a0 x0, a1 x0, a0 x1, a1 x1, a2 x0, a0 x2; the parts of a value that
        // they do not hold (parts_whole) are 0
        uint32_t kept = 0;  // this lane's fragments hold such a value: their last word
#pragma unroll
        for (int m = 0; m < DL_NM; ++m) {
            if (m >= nm) break;
            const uint32_t p0 = pack_bf16x2(ao[m], 0.0f);
            const float r1 = ao[m] - __uint_as_float(p0 << 16);
            const uint32_t p1 = pack_bf16x2(r1, 0.0f);
            const uint32_t p2 = pack_bf16x2(r1 - __uint_as_float(p1 << 16), 0.0f);
            const uint32_t p01 = p0 | (p1 << 16);
            AF[m * KB_BN + tid] = parts_whole(ao[m]) ? uint4{p01, p01, p2 | (p0 << 16), 0u}
                                                     : uint4{0u, 0u, 0u, 1u};
            AO[m * KB_BN + tid] = ao[m];
        }
        // lane lc (hl 0) of wave (wr, wc): row 64 wr + 32 wc + lc, element m its
        // product with member m's factor
        const int32_t xbr = 64 * wr + 32 * wc + lc;
        if (hl == 0) {
            const int32_t m = nm == 1 || xbr >= rows_here ? 0 : tr.member(P, xbr);
            const float v = m == 0 ? xba[0] : m == 1 ? xba[1] : m == 2 ? xba[2] : xba[3];
            const uint32_t p0 = pack_bf16x2(v, 0.0f);
            const float r1 = v - __uint_as_float(p0 << 16);
            const uint32_t p1 = pack_bf16x2(r1, 0.0f);
            const uint32_t p2 = pack_bf16x2(r1 - __uint_as_float(p1 << 16), 0.0f);
            XF[xbr] = parts_whole(v) ? uint4{p0 | (p0 << 16), p1 | (p1 << 16), p0 | (p2 << 16), 0u}
                                     : uint4{0u, 0u, 0u, 1u};
            XB[xbr] = v;
        }
        __syncthreads();
        int32_t rm[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int32_t row = 64 * wr + 32 * i + lc;
            rm[i] = nm == 1 || row >= rows_here ? 0 : tr.member(P, row);
        }
        for (int32_t t = 0; 2 * t < nm; ++t) {
            const int32_t m = 2 * t + hl;  // this lane half's member
            u16x8 xf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                uint4 v = XF[64 * wr + 32 * i + lc];
                kept |= v.w;
                v.w = 0u;
                if (rm[i] != m) v = uint4{0u, 0u, 0u, 0u};
                xf[i] = __builtin_bit_cast(u16x8, v);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint4 v = AF[min(m, nm - 1) * KB_BN + 128 * wc + 32 * j + lc];
                kept |= v.w;
                v.w = 0u;
                const u16x8 af = __builtin_bit_cast(u16x8, v);
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[i][j] = mfma32b(af, xf[i], acc[i][j]);
            }
        }
        if (__ballot(kept != 0) != 0) {
            // outputs with such an operand: the fp32 product (the MFMAs added 0)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float x = XB[64 * wr + 32 * i + lc];
                const bool xw = parts_whole(x);
                const float* ar = AO + rm[i] * KB_BN + 128 * wc + 4 * hl;
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const float f = ar[32 * j + 8 * (e >> 2) + (e & 3)];
                        const float y = __fadd_rn(acc[i][j][e], __fmul_rn(x, f));
                        acc[i][j][e] = xw && parts_whole(f) ? acc[i][j][e] : y;
                        if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // few values live at a time
                    }
            }
        }
    }

    // ---- store -------------------------------------------------------------------------
    // Accumulator element e of lane l is output row lc of the 32-row block and
    // column 8 (e / 4) + 4 hl + e % 4 of the 32-column tile.  Whole aligned tiles go
    // through the wave's own LDS block (the stages are free), 32 rows at a time, so
    // that a store instruction writes 512 (fp32) or 256 (bf16) contiguous bytes per
    // row; the pitch keeps eight lanes' 16-byte accesses on distinct banks.
    constexpr int SP = 528, SPB = 272;  // row pitch in bytes of 128 fp32 / bf16 columns
    const bool whole = vec_y && o0 + KB_BN <= a && (!ybf16 || vec_y == 2);
    unsigned char* sw = smem + wave * 32 * SP;
    if (whole) __syncthreads();  // every wave is past its last LDS read
    auto store_all = [&](auto actc, auto ybc) __attribute__((always_inline)) {
        constexpr int ACT = decltype(actc)::value;
        constexpr bool YB = decltype(ybc)::value;
        if (whole) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int32_t col = 32 * j + 8 * g + 4 * hl;
                        float v[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) v[u] = act_value<ACT>(acc[i][j][4 * g + u]);
                        if constexpr (YB)
                            *reinterpret_cast<uint2*>(sw + lc * SPB + 2 * col) =
                                uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                        else
                            *reinterpret_cast<float4*>(sw + lc * SP + 4 * col) = float4{v[0], v[1], v[2], v[3]};
                    }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                constexpr int RPI = YB ? 4 : 2;            // rows per store instruction
                const int rl = lane / (64 / RPI), cb = lane % (64 / RPI) * 16;
#pragma unroll
                for (int q = 0; q < 32 / RPI; ++q) {
                    const int32_t r32 = q * RPI + rl, row = 64 * wr + 32 * i + r32;
                    const uint4 v = *reinterpret_cast<const uint4*>(sw + r32 * (YB ? SPB : SP) + cb);
                    if (row < rows_here) {
                        const int64_t yoff = row_off(row, P.y_stride, P.y_plane) + o0 + 128 * wc;
                        unsigned char* yp = reinterpret_cast<unsigned char*>(P.y) + yoff * (YB ? 2 : 4) + cb;
                        *reinterpret_cast<uint4*>(yp) = v;
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int32_t row = 64 * wr + 32 * i + lc;
            if (row >= rows_here) continue;
            const int64_t yoff = row_off(row, P.y_stride, P.y_plane) + o0;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int32_t col = 128 * wc + 32 * j + 8 * (e >> 2) + 4 * hl + (e & 3);
                    if (o0 + col >= a) continue;
                    const float v = act_value<ACT>(acc[i][j][e]);
                    if constexpr (YB) reinterpret_cast<uint16_t*>(P.y)[yoff + col] = f2bf(v);
                    else P.y[yoff + col] = v;
                }
        }
    };
    using T0 = std::integral_constant<int, ACT_NONE>;
    using T1 = std::integral_constant<int, ACT_TANH>;
    using T2 = std::integral_constant<int, ACT_SIGMOID>;
    using T3 = std::integral_constant<int, ACT_RELU_SQ>;
    auto by_act = [&](auto ybc) __attribute__((always_inline)) {
        switch (act) {
            case ACT_TANH: store_all(T1{}, ybc); break;
            case ACT_SIGMOID: store_all(T2{}, ybc); break;
            case ACT_RELU_SQ: store_all(T3{}, ybc); break;
            default: store_all(T0{}, ybc); break;
        }
    };
    if (ybf16) by_act(std::true_type{});
    else by_act(std::false_type{});
}

static int32_t bf16_rk(int32_t r) { return r <= 1 ? 1 : 4; }

// Most members a bm-row tile (starting at a multiple of bm) can touch.
static int32_t bf16_nm_max(int32_t bm, int32_t R, int32_t n) {
    int32_t nm;
    if (R % bm == 0) nm = 1;
    else if (R > bm) nm = 2;
    else if (bm % R == 0) nm = bm / R;
    else nm = (bm - 1) / R + 2;
    return std::min(nm, n);
}

static int32_t bf16_kp(int32_t b) { return (b + KB_BK - 1) / KB_BK * KB_BK; }

struct Bf16Plan {
    int32_t rk, nm, bch, kp, bm;
    bool dl;  // the direct-to-LDS pipeline
    size_t lds, w_bytes, f_bytes;
};

static bool bf16_plan(int32_t a, int32_t b, int32_t r, int32_t n, int32_t R, int32_t in_off, Bf16Plan* pl) {
    if (a < KB_BN || b < 1 || n < 1 || r < 0 || r > KB_RMAX || b % 8) return false;
    pl->rk = bf16_rk(r);
    pl->nm = bf16_nm_max(KB_BM, R, n);
    pl->bm = KB_BM;
    pl->kp = bf16_kp(b);
    const size_t bch = r > 0 ? (size_t)pl->nm * (KB_BK / 2) * pl->rk : 0;
    if (bch > (size_t)KB_BPT * KB_THREADS) return false;
    pl->bch = (int32_t)bch;
    const size_t a_lds = r > 0 ? (size_t)pl->nm * KB_BN * pl->rk : 0;
    pl->lds = (size_t)4 * KB_BUF * 2 + (2 * bch + a_lds) * 4;
    // k_gemm_bf16_dl: whole 32-wide K steps, rank 0 or 1 (the factor rows
    // whole groups of four, so that k_factors stores them in 16 and 8 bytes)
    const int32_t nm_dl = bf16_nm_max(DL_BM, R, n);
    pl->dl = b % DL_BK == 0 && pl->rk == 1 &&
             (r == 0 || (nm_dl <= DL_NM && (a + b) % 4 == 0 && in_off % 4 == 0));
    if (pl->dl) {
        pl->nm = nm_dl;
        pl->bm = DL_BM;
        pl->lds = (size_t)DL_NS * DL_SB;
    }
    pl->w_bytes = align16((size_t)a * pl->kp * 2);
    // the factor rows, then at rank 1 room for the input-side ones as bf16
    pl->f_bytes = r > 0 ? align16((size_t)n * (a + b) * r * 4) + (r == 1 ? align16((size_t)n * b * 2) : 0) : 0;
    return true;
}

size_t linear_bf16_workspace(int32_t a, int32_t b, int32_t r, int32_t n, int32_t rows_per_member,
                             int32_t n_time, int32_t math) {
    if (math != HSES_MATH_BF16 || (int64_t)rows_per_member * n_time > INT32_MAX) return 0;
    Bf16Plan pl;
    if (!bf16_plan(a, b, r, n, rows_per_member * n_time, 0, &pl)) return 0;
    return pl.w_bytes + pl.f_bytes;
}

int launch_linear_bf16(LinParams& P, DeviceState* st, hipStream_t s, void* work, size_t work_bytes,
                       int32_t act, int32_t y_fmt) {
    if (P.math != HSES_MATH_BF16) return HSES_ERR_UNSUPPORTED;
    if (P.x_fmt != HSES_FMT_F32 && P.x_fmt != HSES_FMT_BF16) return HSES_ERR_UNSUPPORTED;
    const int32_t r = (P.r > 0 && P.bs != 0.0f) ? P.r : 0;
    Bf16Plan pl;
    if (!bf16_plan(P.a, P.b, r, P.n, P.R, P.tmm ? P.a : 0, &pl) ||
        pl.lds > st->max_lds)
        return HSES_ERR_UNSUPPORTED;
    // 16-byte loads of 8 (bf16) or 4 (fp32) elements: aligned rows, whole groups
    const int64_t vec = P.x_fmt == HSES_FMT_F32 ? 4 : 8;
    if (reinterpret_cast<uintptr_t>(P.x) % 16 || P.x_stride % vec || (P.n_time > 1 && P.x_plane % vec))
        return HSES_ERR_UNSUPPORTED;
    if (!work || work_bytes < pl.w_bytes + pl.f_bytes) return HSES_ERR_UNSUPPORTED;
    const int64_t row_tiles = (P.total + pl.bm - 1) / pl.bm;
    const int64_t tiles = row_tiles * ((P.a + KB_BN - 1) / KB_BN);
    if (tiles > INT32_MAX) return set_error(HSES_ERR_INVALID_ARG, "too many output rows");
    uint16_t* Wb = static_cast<uint16_t*>(work);
    float* F = reinterpret_cast<float*>(static_cast<char*>(work) + pl.w_bytes);
    uint16_t* Fb = reinterpret_cast<uint16_t*>(F) + align16((size_t)P.n * (P.a + P.b) * r * 4) / 2;
    // four consecutive outputs per store (16 bytes fp32, 8 bytes bf16) when every
    // row start keeps them aligned (vec_y 1); bf16 rows 16-byte aligned: eight (2)
    const int64_t ybytes = y_fmt == HSES_FMT_BF16 ? 2 : 4;
    int32_t vec_y = reinterpret_cast<uintptr_t>(P.y) % (4 * ybytes) == 0 && P.y_stride % 4 == 0 &&
                    (P.n_time == 1 || P.y_plane % 4 == 0);
    if (vec_y && ybytes == 2 && reinterpret_cast<uintptr_t>(P.y) % 16 == 0 && P.y_stride % 8 == 0 &&
        (P.n_time == 1 || P.y_plane % 8 == 0))
        vec_y = 2;
    launch_w_to_bf16(P.W, P.a, P.b, pl.kp, P.tmm, Wb, s);
    HSES_CHECK_HIP(hipGetLastError());
    LinParams Q = P;
    Q.r = r;
    if (r > 0) {
        const int rc = launch_factors(Q, st, s, F, pl.dl ? Fb : nullptr);
        if (rc) return rc;
    }
    auto launch = [&](auto kern, int32_t threads, auto... args) -> int {
        HSES_CHECK_HIP(hipFuncSetAttribute((const void*)kern,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds));
        hipLaunchKernelGGL(kern, dim3((uint32_t)tiles), dim3(threads), pl.lds, s, Q, (const uint16_t*)Wb,
                           pl.kp, (const float*)F, args..., act, (int32_t)(y_fmt == HSES_FMT_BF16), vec_y);
        HSES_CHECK_HIP(hipGetLastError());
        return HSES_OK;
    };
    const bool f32 = P.x_fmt == HSES_FMT_F32;
    if (pl.dl)
        return r > 0 ? f32 ? launch(k_gemm_bf16_dl<HSES_FMT_F32, true>, DL_THREADS, (const uint16_t*)Fb)
                           : launch(k_gemm_bf16_dl<HSES_FMT_BF16, true>, DL_THREADS, (const uint16_t*)Fb)
               : f32 ? launch(k_gemm_bf16_dl<HSES_FMT_F32, false>, DL_THREADS, (const uint16_t*)nullptr)
                     : launch(k_gemm_bf16_dl<HSES_FMT_BF16, false>, DL_THREADS, (const uint16_t*)nullptr);
    if (pl.rk == 1)
        return f32 ? launch(k_gemm_bf16<HSES_FMT_F32, 1>, KB_THREADS, pl.bch)
                   : launch(k_gemm_bf16<HSES_FMT_BF16, 1>, KB_THREADS, pl.bch);
    return f32 ? launch(k_gemm_bf16<HSES_FMT_F32, 4>, KB_THREADS, pl.bch)
               : launch(k_gemm_bf16<HSES_FMT_BF16, 4>, KB_THREADS, pl.bch);
}

}  // namespace hses
