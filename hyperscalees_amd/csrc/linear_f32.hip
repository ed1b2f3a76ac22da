// linear_f32.hip -- fp32 perturbed forward y = x W^T + (x B_m) A_m^T for small ranks.
//
// Reference: do_mm_impl (burn_impl/hyperscalees-noiser/src/eggroll.rs:419-446)
// and lora_linear_batched (burn_impl/hyperscalees-models/src/snn.rs:665-685).
//
// Two launches:
//   k_factors   every member's B_m (stream rows [0, b)) and scaled A_m (rows
//             [b, a + b)) into the workspace, each row drawn once; for
//             k_gemm_f32s its last blocks split W into three bf16 parts.
//   k_gemm_f32  y = x W^T with fp32 MFMA (32x32x2) over 128-row x BN-column
//             tiles, K in chunks of 32 staged through double-buffered LDS with
//             the chunk's B_m rows beside them; each thread also accumulates
//             x B_m for its row on the vector ALU from the staged chunk, and the
//             epilogue adds (x B_m) A_m^T with the tile's A_m rows.
//   k_gemm_f32s  the same product on bf16 MFMA (32x32x16) with split operands.
//             An fp32 value is the exact sum of three bf16 parts of 8 significant
//             bits, x = x0 + x1 + x2, so x w needs the six products x0 w0, x0 w1,
//             x1 w0, x1 w1, x0 w2, x2 w0 (the others are below 2^-25 |x w|); bf16
//             activations and spikes are one part: three products.  Products of
//             two parts are exact in the fp32 accumulator.  Six bf16 MFMAs take
//             3/8 of the matrix-core time of the eight fp32 MFMAs they replace:
//             65536 x 1024 -> 1024 at rank 1 (16 rows per member) 1638 -> 855 us,
//             161 TFLOP/s of fp32 product and 964 of issued bf16, against 1144 of a
//             large bf16 product on the same card; error against float64 5.3e-7
//             -> 2.7e-7 (a step of 16 k rounds the leading sum once, not eight
//             times).  Which of the two runs: f32_split_shape.
// The LDS copy of a chunk of k_gemm_f32 stores each row's 32 k values as the
// even k then the odd k, so a lane (row l % 32, k-group l / 32 of the 32x32x2
// MFMA) reads its 16 k-steps of a chunk with four 16-byte loads.
#include <math.h>

#include <type_traits>

#include "linear_common.h"
#include "mfma.h"
#include "noise_dev.h"
#include "runtime.h"

namespace hses {

constexpr int KF_BM = 128, KF_BK = 32, KF_THREADS = 256;
constexpr int KF_XP = 36;          // k_gemm_f32: LDS pitch of a staged row (floats): 16 even k, 16 odd k, pad
constexpr int KF_AMAX = 8192;      // floats of A rows a workgroup keeps for its epilogue
constexpr int KF_RMAX = 16;        // ranks handled
constexpr int KS_BPT = 2;          // k_gemm_f32s: B_m chunk values staged per thread

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x16 mfma32x2(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Value k of row `off` of x in fp32 (k < b checked by the caller).
template <int XFMT>
__device__ __forceinline__ float x_at(const void* x, int64_t off, int32_t k) {
    if constexpr (XFMT == HSES_FMT_BITS) {
        const uint64_t w = static_cast<const uint64_t*>(x)[off + (k >> 6)];
        return (float)((w >> (k & 63)) & 1ull);
    } else if constexpr (XFMT == HSES_FMT_BF16) {
        return bf2f(static_cast<const uint16_t*>(x)[off + k]);
    } else {
        return static_cast<const float*>(x)[off + k];
    }
}

// Item i of the split of W: a piece of 8 k of one output row.
__device__ __forceinline__ void split_w(const LinParams& P, uint16_t* Wp, int32_t a_pad, int64_t i) {
    const int32_t nch = (P.b + KF_BK - 1) / KF_BK;
    if (i >= (int64_t)nch * a_pad * 4) return;
    // consecutive lanes: the pieces of a row (W rows contiguous in k), or for
    // do_Tmm the output rows (W columns contiguous in the output)
    const int32_t ch = (int32_t)(i / (a_pad * 4)), e = (int32_t)(i - (int64_t)ch * a_pad * 4);
    const int32_t o = P.tmm ? e % a_pad : e >> 2, pc = P.tmm ? e / a_pad : e & 3;
    const int32_t k0 = ch * KF_BK + 8 * pc;
    const int64_t w0 = P.tmm ? (int64_t)k0 * P.a + o : (int64_t)o * P.b + k0;
    const int64_t wk = P.tmm ? P.a : 1;
    uint32_t d[3][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const bool ok = o < P.a;
        const float lo = ok && k0 + 2 * u < P.b ? P.W[w0 + 2 * u * wk] : 0.0f;
        const float hi = ok && k0 + 2 * u + 1 < P.b ? P.W[w0 + (2 * u + 1) * wk] : 0.0f;
        uint32_t p[3];
        split3(lo, hi, p);
#pragma unroll
        for (int w = 0; w < 3; ++w) d[w][u] = p[w];
    }
#pragma unroll
    for (int w = 0; w < 3; ++w)
        reinterpret_cast<uint4*>(Wp)[((int64_t)(ch * 3 + w) * a_pad + o) * 4 + slot_of(o, pc)] =
            uint4{d[w][0], d[w][1], d[w][2], d[w][3]};
}

// ---- k_factors -------------------------------------------------------------------
// F[m] = the member's (a + b) x r stream rows as drawn, except that the
// rows carrying sign * sigma / sqrt(r) are scaled: do_mm's A rows [b, a + b),
// do_Tmm's input-side rows [a, a + b) (with a the output width).  Members 2p
// and 2p + 1 share pair p's normals with the scaled rows negated, so a thread
// draws rows [q rc, q rc + rc) of one pair after one jump to the group's start
// and stores them for both members.  Bound by the draw's vector instructions
// (about 106 per normal): drawing per pair and not per member halves them
// (4096 members, 2048 rows, rank 1: 42.8 -> 37 us).
// Blocks from fblocks on split W for k_gemm_f32s (Wp, NULL without one): with
// a_pad output rows, [k chunk of 32][part][output row][32], the 16-byte pieces
// of a row swizzled as k_gemm_f32s reads them from LDS (slot_of), zero past a
// and b.  A block takes 256 pieces of 8 k.
// vec: every group starts 16-byte aligned.  Fb (rank 1, or NULL): the input-side
// rows go there as bf16, [member][b], instead of into F.
__global__ __launch_bounds__(256) void k_factors(LinParams P, int32_t rc, int32_t groups, int32_t pairs,
                                                 float* __restrict__ F, uint16_t* __restrict__ Fb,
                                                 int32_t vec, int32_t fblocks,
                                                 uint16_t* __restrict__ Wp, int32_t a_pad) {
    __shared__ BmTables t;
    if ((int32_t)blockIdx.x >= fblocks) {
        split_w(P, Wp, a_pad, (int64_t)(blockIdx.x - fblocks) * 256 + threadIdx.x);
        return;
    }
    load_bm_tables(&t, P.tables);
    __syncthreads();
    const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (item >= (int64_t)pairs * groups) return;
    const int32_t p = (int32_t)(item / groups), q = (int32_t)(item % groups);
    const int32_t r = P.r, rows = P.a + P.b, row0 = q * rc;
    const int32_t tid = 2 * (P.tid_lo / 2 + p), m = tid - P.tid_lo;  // the pair's even member (-1: not ours)
    float sign;
    const uint64_t seed = member_seed(P.key, P.epoch, P.nreuse, tid, &sign);
    uint64_t s = row_start_state(seed, q, P.jump);
    const NoiseCtx ctx{&t, P.log_exc, P.cos_exc};
    float* even = F + ((int64_t)m * rows + row0) * r;
    float* odd = even + (int64_t)rows * r;
    const bool we = m >= 0, wo = m + 1 < P.n;
    const int32_t split = ((P.tmm ? P.a : P.b) - row0) * r;  // normals before the first scaled row
    const int32_t k0 = row0 - (P.tmm ? P.a : 0);             // input row of normal 0 (rank 1)
    auto one = [&](int32_t i, float v) {
        const float e = i >= split ? v * P.bs : v;
        if (Fb && k0 + i >= 0 && k0 + i < P.b) {
            uint16_t* fb = Fb + (int64_t)m * P.b + k0 + i;
            if (we) fb[0] = f2bf(e);
            if (wo) fb[P.b] = f2bf(i >= split ? -e : e);
            return;
        }
        if (we) even[i] = e;
        if (wo) odd[i] = i >= split ? -e : e;
    };
    bm_run2<4>(
        s, min(rc, rows - row0) * r, ctx,
        [&](int32_t i, const float* v) {
            if (!vec) {
#pragma unroll
                for (int u = 0; u < 4; ++u) one(i + u, v[u]);
                return;
            }
            float4 e, o;
            float* ep = reinterpret_cast<float*>(&e);
            float* op = reinterpret_cast<float*>(&o);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool sc = i + u >= split;
                ep[u] = sc ? v[u] * P.bs : v[u];
                op[u] = sc ? -ep[u] : ep[u];
            }
            if (Fb && k0 + i >= 0 && k0 + i < P.b) {
                uint16_t* fb = Fb + (int64_t)m * P.b + k0 + i;
                if (we) *reinterpret_cast<uint2*>(fb) = uint2{pack_bf16x2(e.x, e.y), pack_bf16x2(e.z, e.w)};
                if (wo)
                    *reinterpret_cast<uint2*>(fb + P.b) = uint2{pack_bf16x2(o.x, o.y), pack_bf16x2(o.z, o.w)};
                return;
            }
            if (we) *reinterpret_cast<float4*>(even + i) = e;
            if (wo) *reinterpret_cast<float4*>(odd + i) = o;
        },
        one);
}

// ---- k_gemm_f32s -----------------------------------------------------------------
// What bounds it: the matrix cores.  The x chunk goes global -> registers (one
// chunk ahead) -> three parts in LDS, W arrives split (its conversion would
// repeat in every row tile); 48 KB of LDS and two waves per SIMD let two
// workgroups share a CU, one's conversion and barriers beside the other's MFMAs.
// A BM x BN tile, four waves: 2 x 2 of (BM / 2) x 64 for BN = 128, 2 x 2 of 32 x 32
// for 64 x 64, else four of 32 rows.  RK is the rank padded to 1, 4, 8 or 16
// (the LDS copies of B_m and A_m rows hold RK values per row, zero past r).
template <int XFMT, int BM, int BN, int RK>
__global__ __launch_bounds__(KF_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_f32s(LinParams P, const float* __restrict__ F, const uint16_t* __restrict__ Wp, int32_t a_pad,
                 int32_t bch) {
    constexpr bool SQ = BN == 128 || BM == 64;          // 2 x 2 waves
    constexpr int WM = SQ ? BM / 2 : 32, WN = SQ ? BN / 2 : BN;
    constexpr int MI = WM / 32, NJ = WN / 32;           // 32 x 32 MFMA tiles of a wave
    constexpr int NP = XFMT == HSES_FMT_F32 ? 3 : 1;    // parts of x
    constexpr bool XLDS = XFMT != HSES_FMT_BITS;        // bits are expanded from registers
    constexpr int TPR = KF_THREADS / BM, KPT = KF_BK / TPR;  // threads per x row, k per thread
    extern __shared__ __align__(16) unsigned char smem[];
    // x parts [NP][BM][32], W parts [3][BN][32] (bf16, 64-byte rows, pieces
    // swizzled by slot_of), the chunk's B_m rows [lm][32][RK], the tile's A_m
    // rows [lm][BN][RK], then per row the y and x offsets and the member.
    uint16_t* Xs = reinterpret_cast<uint16_t*>(smem);
    uint16_t* Ws = Xs + (XLDS ? NP * BM * KF_BK : 0);
    float* Bc = reinterpret_cast<float*>(Ws + 3 * BN * KF_BK);
    int64_t* yoffs = reinterpret_cast<int64_t*>(Bc + bch);
    int64_t* xoffs = yoffs + BM;
    int32_t* rlm = reinterpret_cast<int32_t*>(xoffs + BM);
    float* As = reinterpret_cast<float*>(rlm + BM);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t lc = lane & 31, kh = lane >> 5;
    const int wm0 = SQ ? (wave >> 1) * WM : wave * 32, wn0 = SQ ? (wave & 1) * WN : 0;
    // Tile of this workgroup: workgroups are dealt to the 8 XCDs in turn, so
    // XCD x gets the contiguous tile range x * nb / 8 .. with the column tiles
    // of a row tile adjacent: the workgroups that read the same x rows run on
    // one XCD together and share its L2.
    int64_t L0;
    int32_t o0;
    {
        const uint32_t nb = gridDim.x, g = blockIdx.x, xcd = g & 7u, j = g >> 3;
        const uint32_t q = nb >> 3, rem = nb & 7u;
        const uint32_t ncol = (uint32_t)((P.a + BN - 1) / BN);
        const uint32_t t = ncol == 1 ? g  // one column tile: no x rows are shared
                           : xcd < rem ? xcd * (q + 1) + j : rem * (q + 1) + (xcd - rem) * q + j;
        L0 = (int64_t)(t / ncol) * BM;
        o0 = (int32_t)(t % ncol) * BN;
    }
    const int32_t ct = min(BN, P.a - o0);
    const int32_t r = P.r, b = P.b;
    const int32_t rows_here = (int32_t)min<int64_t>(BM, P.total - L0);
    const TileRows tr(P, L0);
    const int32_t nm = tr.member(P, rows_here - 1) + 1;
    const bool noisy = r > 0;
    const int64_t fpitch = (int64_t)(P.a + b) * r;  // floats of one member's factors
    const float* Fm = F + (int64_t)tr.m_first * fpitch;
    const int32_t in_off = P.tmm ? P.a : 0, out_off = P.tmm ? 0 : b;  // factor rows by role

    if (tid < BM) {
        const bool ok = tid < rows_here;
        yoffs[tid] = ok ? tr.offset(P, tid, P.y_stride, P.y_plane) + o0 : 0;
        xoffs[tid] = ok ? tr.offset(P, tid, P.x_stride, P.x_plane) : 0;
        rlm[tid] = ok ? tr.member(P, tid) : 0;
    }
    // ---- the output-side factor rows of the tile's members -----------------------
    if (noisy) {
        for (int32_t i = tid; i < nm * BN * RK; i += KF_THREADS) {
            const int32_t c = i % RK, o = (i / RK) % BN, lm = i / (RK * BN);
            As[i] = (c < r && o < ct) ? Fm[lm * fpitch + (int64_t)(out_off + o0 + o) * r + c] : 0.0f;
        }
    }
    __syncthreads();

    // ---- staging: thread -> x row tid / TPR (KPT k), BN * 3 / 64 pieces of W ---------
    const int xr = tid / TPR, xk = (tid % TPR) * KPT;
    const bool xvalid = xr < rows_here;
    const int64_t xoff = xoffs[xr];
    const int32_t xlm = rlm[xr];
    const bool xal = (reinterpret_cast<uintptr_t>(P.x) & 15) == 0 &&
                     (xoff & (XFMT == HSES_FMT_F32 ? 3 : 7)) == 0;  // 16-byte loads
    constexpr int WPC = (BN * 12 + KF_THREADS - 1) / KF_THREADS;  // 16-byte pieces per thread
    constexpr int BPT = KS_BPT;  // B_m chunk values per thread
    float xv[KPT];
    u32x4 wv[WPC];
    uint32_t xw[MI], xbits = 0;  // bit-packed x: the chunk of the MFMA rows, of row xr
    float bv[BPT];
    int64_t xwo[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) xwo[i] = XLDS ? 0 : 2 * xoffs[wm0 + 32 * i + lc];
    // B_m chunk value j: [lm][kk][c], its float offset from Fm at chunk 0
    int32_t boff[BPT], bkk[BPT];
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        const int32_t e = tid + KF_THREADS * j;
        const int32_t c = e % RK, kk = (e / RK) % KF_BK, lm = e / (RK * KF_BK);
        bkk[j] = (e < bch && lm < nm && c < r) ? kk : b;  // b: never valid
        boff[j] = (int32_t)(lm * fpitch) + (in_off + kk) * r + c;
    }
    auto b_ok = [&](int j, int32_t kc) { return kc * KF_BK + bkk[j] < b; };
    auto load_chunk = [&](int32_t kc) {
        const int32_t k = kc * KF_BK + xk;
        if constexpr (!XLDS) {
            const uint32_t* xp = static_cast<const uint32_t*>(P.x);
#pragma unroll
            for (int i = 0; i < MI; ++i)
                xw[i] = wm0 + 32 * i + lc < rows_here ? xp[xwo[i] + kc] : 0u;
            if (noisy) xbits = xvalid ? xp[2 * xoff + kc] >> xk : 0u;
        } else if (xvalid && xal && k + KPT <= b) {
            if constexpr (XFMT == HSES_FMT_F32) {
                const float4* xp = reinterpret_cast<const float4*>(static_cast<const float*>(P.x) + xoff + k);
#pragma unroll
                for (int q = 0; q < KPT / 4; ++q) *reinterpret_cast<float4*>(xv + 4 * q) = xp[q];
            } else {
                const uint4* xp = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(P.x) + xoff + k);
#pragma unroll
                for (int q = 0; q < KPT / 8; ++q) {
                    const uint4 u = xp[q];
                    const uint32_t w4[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        xv[8 * q + 2 * e] = __uint_as_float(w4[e] << 16);
                        xv[8 * q + 2 * e + 1] = __uint_as_float(w4[e] & 0xffff0000u);
                    }
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < KPT; ++i)
                xv[i] = (xvalid && k + i < b) ? x_at<XFMT>(P.x, xoff, k + i) : 0.0f;
        }
        // W parts of the chunk: [part][o0 ..][32], whole 64-byte rows
#pragma unroll
        for (int j = 0; j < WPC; ++j) {
            const int32_t e = tid + KF_THREADS * j, p = e / (BN * 4), q = e % (BN * 4);
            if (BN * 12 % KF_THREADS == 0 || e < BN * 12)
                wv[j] = reinterpret_cast<const u32x4*>(Wp)[((int64_t)(kc * 3 + p) * a_pad + o0) * 4 + q];
        }
        if (noisy) {
#pragma unroll
            for (int j = 0; j < BPT; ++j)
                if (KF_THREADS * j < bch)  // uniform
                    bv[j] = Fm[b_ok(j, kc) ? boff[j] + kc * KF_BK * r : 0];
        }
    };
    auto store_chunk = [&](int32_t kc) {
#pragma unroll
        for (int q = 0; q < (XLDS ? KPT / 8 : 0); ++q) {
            uint32_t d[3][4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                uint32_t p[3];
                const float lo = xv[8 * q + 2 * u], hi = xv[8 * q + 2 * u + 1];
                if constexpr (NP == 3) split3(lo, hi, p);
                else p[0] = (__float_as_uint(lo) >> 16) | (__float_as_uint(hi) & 0xffff0000u);
#pragma unroll
                for (int w = 0; w < NP; ++w) d[w][u] = p[w];
            }
            const int s = slot_of(xr, (xk >> 3) + q);
#pragma unroll
            for (int w = 0; w < NP; ++w)
                *reinterpret_cast<uint4*>(Xs + (w * BM + xr) * KF_BK + 8 * s) =
                    uint4{d[w][0], d[w][1], d[w][2], d[w][3]};
        }
#pragma unroll
        for (int j = 0; j < WPC; ++j) {
            const int32_t e = tid + KF_THREADS * j;
            if (BN * 12 % KF_THREADS == 0 || e < BN * 12) reinterpret_cast<u32x4*>(Ws)[e] = wv[j];
        }
        if (noisy) {
#pragma unroll
            for (int j = 0; j < BPT; ++j) {
                const int32_t e = tid + KF_THREADS * j;
                if (KF_THREADS * j < bch && e < bch) Bc[e] = b_ok(j, kc) ? bv[j] : 0.0f;
            }
        }
    };

    // acc: the products of the leading parts; low: those of the others, 2^-8 of
    // them and less, so that the rounding of their many sums does not count
    f32x16 acc[MI][NJ], low[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = low[i][j][e] = 0.0f;
    float xb[RK];  // this thread's share of (x B_m) for row xr
#pragma unroll
    for (int c = 0; c < RK; ++c) xb[c] = 0.0f;

    const int32_t nch = (b + KF_BK - 1) / KF_BK;
    load_chunk(0);
    for (int32_t kc = 0; kc < nch; ++kc) {
        if (kc) __syncthreads();  // every wave is past its reads of chunk kc - 1
        store_chunk(kc);
        __syncthreads();
        if (noisy) {
            // x B_m over this thread's KPT k, fp32 in ascending k
            const float* bs = Bc + (xlm * KF_BK + xk) * RK;
#pragma unroll
            for (int i = 0; i < KPT; ++i) {
                float be[RK];
                if constexpr (RK == 1) {
                    be[0] = bs[i];
                } else {
#pragma unroll
                    for (int q = 0; q < RK / 4; ++q)
                        *reinterpret_cast<float4*>(be + 4 * q) =
                            *reinterpret_cast<const float4*>(bs + i * RK + 4 * q);
                }
                const float v = XLDS ? xv[i] : (float)((xbits >> i) & 1u);
#pragma unroll
                for (int c = 0; c < RK; ++c) xb[c] = __builtin_fmaf(v, be[c], xb[c]);
            }
        }
        uint32_t xc[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i) xc[i] = XLDS ? 0u : xw[i];
        if (kc + 1 < nch) load_chunk(kc + 1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            u16x8 af[MI][NP], bf[NJ][3];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int row = wn0 + 32 * j + lc, s = slot_of(row, 2 * ks + kh);
#pragma unroll
                for (int p = 0; p < 3; ++p) bf[j][p] = lds_u16x8(Ws + (p * BN + row) * KF_BK + 8 * s);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                if constexpr (XLDS) {
                    const int row = wm0 + 32 * i + lc, s = slot_of(row, 2 * ks + kh);
#pragma unroll
                    for (int p = 0; p < NP; ++p) af[i][p] = lds_u16x8(Xs + (p * BM + row) * KF_BK + 8 * s);
                } else {
                    af[i][0] = expand_bits((xc[i] >> (16 * ks + 8 * kh)) & 0xffu);
                }
            }
            // the products down to 2^-16 of the largest: x_p w_q, p + q <= 2
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int q = 0; q < 3 - p; ++q)
#pragma unroll
                    for (int i = 0; i < MI; ++i)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            if (p + q == 0) acc[i][j] = mfma_bf(af[i][p], bf[j][q], acc[i][j]);
                            else low[i][j] = mfma_bf(af[i][p], bf[j][q], low[i][j]);
                        }
        }
    }

    // ---- epilogue: y = x W^T + (x B_m) A_m^T -----------------------------------------
    __syncthreads();
    float* XBs = reinterpret_cast<float*>(smem);  // [BM][RK]; the staging buffers are free
    if (noisy) {
#pragma unroll
        for (int c = 0; c < RK; ++c) {
            float v = xb[c] + __shfl_xor(xb[c], 1);  // the row's k shares
            if constexpr (TPR == 4) v += __shfl_xor(v, 2);
            if (xk == 0) XBs[xr * RK + c] = v;
        }
        __syncthreads();
    }
    auto add_noise = [&](float yv, int32_t row, int32_t col) {
        const float* ar = As + ((size_t)rlm[row] * BN + col) * RK;
        float z = 0.0f;
#pragma unroll
        for (int c = 0; c < RK; ++c) z = __fadd_rn(z, __fmul_rn(XBs[row * RK + c], ar[c]));
        return __fadd_rn(yv, z);
    };
    // accumulator element e of lane l: row 8 (e / 4) + 4 kh + e % 4 of the
    // 32-row tile, column lc
    auto past = [](float v) {
        const float a = fabsf(v);
        return !(a < INFINITY) || (a < 0x1p-60f && a > 0.0f);
    };
    // the largest of (bits of |sum|) - (bits of 2^-60), doubled: one of a sum past either
    // bound, or of 0, is at least that of infinity
    constexpr uint32_t kLow = 0x21800000u << 1, kInf = 0x7f800000u << 1;
    uint32_t far = 0;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int32_t row = wm0 + 32 * i + 8 * (e >> 2) + 4 * kh + (e & 3);
            if (row >= rows_here) continue;
            float* yrow = P.y + yoffs[row];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int32_t col = wn0 + 32 * j + lc;
                if (col >= ct) continue;
                const float yv = __fadd_rn(acc[i][j][e], low[i][j][e]);
                far = max(far, (__float_as_uint(yv) << 1) - kLow);
                yrow[col] = noisy ? add_noise(yv, row, col) : yv;
            }
        }
    // A part of an infinity, a NaN or a magnitude that rounds up to infinity is not
    // finite and leaves its row or column of sums so.  Parts below 2^-126 lose bits
    // (operands under 2^-102, split3): b 2^-126 times the other operand, less than
    // the fp32 sums' own rounding where |y| >= 2^-60 and the operands are below 2^42.
    // Outputs past either bound are formed again with plain fp32 chains, which give what
    // fp32 gives (sums of exactly 0, as of rows of zeros, stand), each by its lane, so
    // that rows of small values do not slow down the others (16384 x 1024 -> 1024 with
    // one row in 128 scaled by 2^-80: 0.55 ms, and 21 with the wave's outputs; 0.26
    // without such rows).
    if (!__any(far >= kInf - kLow)) return;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            uint32_t left = 0;  // this lane's outputs of the 32 x 32 tile, a bit each
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int32_t row = wm0 + 32 * i + 8 * (e >> 2) + 4 * kh + (e & 3);
                if (row < rows_here && past(__fadd_rn(acc[i][j][e], low[i][j][e]))) left |= 1u << e;
            }
            const int32_t col = wn0 + 32 * j + lc;
            if (col >= ct) left = 0;
            const float* w = P.W + (P.tmm ? o0 + col : (int64_t)(o0 + col) * b);
            const int64_t wk = P.tmm ? P.a : 1;
#pragma unroll 1
            for (; left; left &= left - 1) {
                const int32_t e = __builtin_ctz(left);
                const int32_t row = wm0 + 32 * i + 8 * (e >> 2) + 4 * kh + (e & 3);
                const int64_t xo = xoffs[row];
                float yv = 0.0f;
#pragma unroll 1
                for (int32_t k = 0; k < b; ++k) yv = __builtin_fmaf(x_at<XFMT>(P.x, xo, k), w[k * wk], yv);
                P.y[yoffs[row] + col] = noisy ? add_noise(yv, row, col) : yv;
            }
        }
}

// ---- k_gemm_f32 ------------------------------------------------------------------
// The epilogue keeps the A_m rows as [member][RK / 4][column][4] in LDS, so that the
// 32 columns of a 16-byte read fall on distinct banks (as rows of RK they shared
// eight: 70% of the kernel's LDS cycles at 16 -> 64, rank 8), reads them once when
// the tile has one member, and takes each row's offset and member from an LDS
// table (the divisions of 16 rows per lane were most of its vector instructions).
// Bits do not change.  Whole calls: 524288 x 16 -> 64 at rank 8 168 -> 83 us, spike rows at
// rank 4 131072 x 128 -> 128 84 -> 73 and 131072 x 784 -> 128 316 -> 305 (its MFMAs bound
// it), 32768 spike rows 200 -> 200 at rank 8 and 16 rows a member 89 -> 64.
//
// NT 32-column MFMA tiles per wave (BN = 32 NT); four waves of 32 rows.  RK is
// the rank padded to 1, 4, 8 or 16 (the LDS copies of B_m and A_m rows hold RK
// values per row, zero past r).
template <int XFMT, int NT, int RK>
__global__ __launch_bounds__(KF_THREADS) void k_gemm_f32(LinParams P, const float* __restrict__ F,
                                                         int32_t bch, int32_t nm_max) {
    constexpr int BN = 32 * NT;
    extern __shared__ __align__(16) unsigned char smem[];
    // Two staging buffers, each: 128 x rows, BN W rows (KF_XP floats each), then
    // the chunk's B_m rows of the tile's members ([lm][32][RK]).  After them the
    // tile's A_m rows ([lm][RK / 4][BN][4]) and each row's y offset and member.  bch
    // (floats of a chunk's B_m rows, 0 without noise) and nm_max (members a tile can
    // touch) are the host's, which sized the LDS.
    const int32_t bufsz = (KF_BM + BN) * KF_XP + bch;
    float* buf = reinterpret_cast<float*>(smem);
    // one staging buffer when K is a single chunk (b <= 32), else two
    float* As = buf + (P.b > KF_BK ? 2 : 1) * bufsz;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t lc = lane & 31, kh = lane >> 5;
    // Tile of this workgroup: workgroups are dealt to the 8 XCDs in turn, so
    // XCD x gets the contiguous tile range x * nb / 8 .. with the column tiles
    // of a row tile adjacent: the workgroups that read the same x rows run on
    // one XCD together and share its L2.
    int64_t L0;
    int32_t o0;
    {
        const uint32_t nb = gridDim.x, g = blockIdx.x, xcd = g & 7u, j = g >> 3;
        const uint32_t q = nb >> 3, rem = nb & 7u;
        const uint32_t ncol = (uint32_t)((P.a + BN - 1) / BN);
        const uint32_t t = ncol == 1 ? g  // one column tile: no x rows are shared
                           : xcd < rem ? xcd * (q + 1) + j : rem * (q + 1) + (xcd - rem) * q + j;
        L0 = (int64_t)(t / ncol) * KF_BM;
        o0 = (int32_t)(t % ncol) * BN;
    }
    const int32_t ct = min(BN, P.a - o0);
    const int32_t r = P.r, b = P.b;
    const int32_t rows_here = (int32_t)min<int64_t>(KF_BM, P.total - L0);
    const TileRows tr(P, L0);
    const int32_t m_first = tr.m_first;
    const int32_t nm = tr.member(P, rows_here - 1) + 1;
    const bool noisy = r > 0;
    const int64_t fpitch = (int64_t)(P.a + b) * r;  // floats of one member's factors
    const float* Fm = F + (int64_t)m_first * fpitch;
    int64_t* yoffs = reinterpret_cast<int64_t*>(As + (noisy ? nm_max * BN * RK : 0));
    int32_t* rlm = reinterpret_cast<int32_t*>(yoffs + KF_BM);
    if (tid < KF_BM) {
        const bool ok = tid < rows_here;
        yoffs[tid] = ok ? tr.offset(P, tid, P.y_stride, P.y_plane) + o0 : 0;
        rlm[tid] = ok ? tr.member(P, tid) : 0;
    }

    // ---- A rows of the tile's members: F rows b + o0 .. b + o0 + ct ------------
    constexpr int RQ = RK < 4 ? 1 : RK / 4, RC = RK < 4 ? RK : 4;  // [lm][RQ][BN][RC]
    if (noisy) {
        for (int32_t i = tid; i < nm * BN * RK; i += KF_THREADS) {
            const int32_t c = i % RK, o = (i / RK) % BN, lm = i / (RK * BN);
            As[((lm * RQ + c / RC) * BN + o) * RC + c % RC] =
                (c < r && o < ct) ? Fm[lm * fpitch + (int64_t)(b + o0 + o) * r + c] : 0.0f;
        }
    }

    // ---- staging: thread -> x row tid / 2 (16 k), W row tid * BN / 256 ----------
    const int xr = tid >> 1, xk = (tid & 1) * 16;
    const int64_t Lx = L0 + xr;
    const bool xvalid = Lx < P.total;
    const int64_t xoff = xvalid ? tr.offset(P, xr, P.x_stride, P.x_plane) : 0;
    const int32_t xlm = xvalid ? tr.member(P, xr) : 0;  // the x row's member in the tile
    constexpr int WPT = BN * KF_BK / KF_THREADS;  // W values per thread: 16, 8 or 4
    constexpr int WTPR = KF_BK / WPT;             // threads per W row
    const int wr = tid / WTPR, wk = (tid % WTPR) * WPT;
    const int32_t wo = o0 + wr;
    const bool wvalid = wo < P.a;
    const float* wrow = P.W + (size_t)(wvalid ? wo : 0) * b;
    constexpr int BPT = 8;  // B_m chunk values per thread (bch <= 8 * 256)
    float xv[16], wv[WPT], bv[BPT];
    auto load_chunk = [&](int32_t k0) {
        if constexpr (XFMT == HSES_FMT_BITS) {
            uint32_t bits = 0;
            const int32_t k = k0 + xk;
            if (xvalid && k < b) {
                const uint64_t w = static_cast<const uint64_t*>(P.x)[xoff + (k >> 6)];
                bits = (uint32_t)(w >> (k & 63)) & 0xffffu;
                if (b - k < 16) bits &= (1u << (b - k)) - 1u;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) xv[i] = (float)((bits >> i) & 1u);
        } else {
            const int32_t k = k0 + xk;
            bool vec = xvalid && k + 16 <= b;
            if constexpr (XFMT == HSES_FMT_F32) {
                const float* xp = static_cast<const float*>(P.x) + xoff + k;
                if (vec && (reinterpret_cast<uintptr_t>(xp) & 15) == 0) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<float4*>(xv + 4 * q) = reinterpret_cast<const float4*>(xp)[q];
                } else {
                    vec = false;
                }
            } else {
                const uint16_t* xp = static_cast<const uint16_t*>(P.x) + xoff + k;
                if (vec && (reinterpret_cast<uintptr_t>(xp) & 15) == 0) {
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const uint4 u = reinterpret_cast<const uint4*>(xp)[q];
                        const uint32_t w4[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            xv[8 * q + 2 * e] = __uint_as_float(w4[e] << 16);
                            xv[8 * q + 2 * e + 1] = __uint_as_float(w4[e] & 0xffff0000u);
                        }
                    }
                } else {
                    vec = false;
                }
            }
            if (!vec) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    xv[i] = (xvalid && k + i < b) ? x_at<XFMT>(P.x, xoff, k + i) : 0.0f;
            }
        }
        {
            const int32_t k = k0 + wk;
            const float* wp = wrow + k;
            if (wvalid && k + WPT <= b && (reinterpret_cast<uintptr_t>(wp) & 15) == 0) {
#pragma unroll
                for (int q = 0; q < WPT / 4; ++q)
                    *reinterpret_cast<float4*>(wv + 4 * q) = reinterpret_cast<const float4*>(wp)[q];
            } else {
#pragma unroll
                for (int i = 0; i < WPT; ++i) wv[i] = (wvalid && k + i < b) ? wp[i] : 0.0f;
            }
        }
        if (noisy) {
#pragma unroll
            for (int j = 0; j < BPT; ++j) {
                const int32_t e = tid + KF_THREADS * j;  // [lm][kk][c] of the chunk
                const int32_t c = e % RK, kk = (e / RK) % KF_BK, lm = e / (RK * KF_BK);
                bv[j] = (e < bch && lm < nm && c < r && k0 + kk < b)
                            ? Fm[lm * fpitch + (int64_t)(k0 + kk) * r + c]
                            : 0.0f;
            }
        }
    };
    // even k to [0, 16), odd k to [16, 32) of the row, by k / 2
    auto store_chunk = [&](float* B) {
        float* xd = B + xr * KF_XP + (xk >> 1);
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            xd[i >> 1] = xv[i];
            xd[16 + (i >> 1)] = xv[i + 1];
        }
        float* wd = B + (KF_BM + wr) * KF_XP + (wk >> 1);
#pragma unroll
        for (int i = 0; i < WPT; i += 2) {
            wd[i >> 1] = wv[i];
            wd[16 + (i >> 1)] = wv[i + 1];
        }
        if (noisy) {
            float* bd = B + (KF_BM + BN) * KF_XP;
#pragma unroll
            for (int j = 0; j < BPT; ++j) {
                const int32_t e = tid + KF_THREADS * j;
                if (e < bch) bd[e] = bv[j];
            }
        }
    };

    f32x16 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
    float xb[RK];  // this thread's half of (x B_m) for row xr
#pragma unroll
    for (int c = 0; c < RK; ++c) xb[c] = 0.0f;

    const int32_t nch = (b + KF_BK - 1) / KF_BK;
    load_chunk(0);
    store_chunk(buf);
    __syncthreads();
    for (int32_t kc = 0; kc < nch; ++kc) {
        const float* B = buf + (kc & 1) * bufsz;
        if (kc + 1 < nch) load_chunk((kc + 1) * KF_BK);
        const float* ap = B + (wave * 32 + lc) * KF_XP + 16 * kh;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            float af[8], bfr[NT][8];
            *reinterpret_cast<float4*>(af) = *reinterpret_cast<const float4*>(ap + 8 * half);
            *reinterpret_cast<float4*>(af + 4) = *reinterpret_cast<const float4*>(ap + 8 * half + 4);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const float* bp = B + (KF_BM + 32 * j + lc) * KF_XP + 16 * kh + 8 * half;
                *reinterpret_cast<float4*>(bfr[j]) = *reinterpret_cast<const float4*>(bp);
                *reinterpret_cast<float4*>(bfr[j] + 4) = *reinterpret_cast<const float4*>(bp + 4);
            }
#pragma unroll
            for (int s = 0; s < 8; ++s)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[j] = mfma32x2(af[s], bfr[j][s], acc[j]);
        }
        if (noisy) {
            // x B_m over this thread's 16 k: even k xk + 2 i at [xk / 2 + i], odd at 16 + ..
            const float* xs = B + xr * KF_XP + (xk >> 1);
            const float* bs = B + (KF_BM + BN) * KF_XP + (xlm * KF_BK + xk) * RK;
            float ev[8], od[8];
            *reinterpret_cast<float4*>(ev) = *reinterpret_cast<const float4*>(xs);
            *reinterpret_cast<float4*>(ev + 4) = *reinterpret_cast<const float4*>(xs + 4);
            *reinterpret_cast<float4*>(od) = *reinterpret_cast<const float4*>(xs + 16);
            *reinterpret_cast<float4*>(od + 4) = *reinterpret_cast<const float4*>(xs + 20);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float be[RK], bo[RK];
                if constexpr (RK == 1) {
                    be[0] = bs[2 * i];
                    bo[0] = bs[2 * i + 1];
                } else {
#pragma unroll
                    for (int q = 0; q < RK / 4; ++q) {
                        *reinterpret_cast<float4*>(be + 4 * q) =
                            *reinterpret_cast<const float4*>(bs + (2 * i) * RK + 4 * q);
                        *reinterpret_cast<float4*>(bo + 4 * q) =
                            *reinterpret_cast<const float4*>(bs + (2 * i + 1) * RK + 4 * q);
                    }
                }
#pragma unroll
                for (int c = 0; c < RK; ++c) {
                    xb[c] = __builtin_fmaf(ev[i], be[c], xb[c]);
                    xb[c] = __builtin_fmaf(od[i], bo[c], xb[c]);
                }
            }
        }
        if (kc + 1 < nch) store_chunk(buf + ((kc + 1) & 1) * bufsz);
        __syncthreads();
    }

    // ---- epilogue: y = x W^T + (x B_m) A_m^T -----------------------------------
    float* XBs = buf;  // [128][RK]; the staging buffers are free after the last barrier
    if (noisy) {
#pragma unroll
        for (int c = 0; c < RK; ++c) {
            const float v = xb[c] + __shfl_xor(xb[c], 1);  // the row's two k halves
            if (xk == 0) XBs[xr * RK + c] = v;
        }
        __syncthreads();
    }
    // accumulator element e of lane l: row 8 (e / 4) + 4 kh + e % 4 of the
    // wave's 32, column lc of the tile
    float ar[NT][RK];
    auto load_a = [&](int32_t lm) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < RQ; ++q) {
                const float* p = As + ((lm * RQ + q) * BN + 32 * j + lc) * RC;
                if constexpr (RC == 4) {
                    const float4 v = *reinterpret_cast<const float4*>(p);
                    ar[j][4 * q] = v.x, ar[j][4 * q + 1] = v.y, ar[j][4 * q + 2] = v.z, ar[j][4 * q + 3] = v.w;
                } else {
                    ar[j][0] = p[0];
                }
            }
    };
    if (noisy && nm == 1) load_a(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int32_t row = wave * 32 + 8 * (e >> 2) + 4 * kh + (e & 3);
        if (row >= rows_here) continue;
        float* yrow = P.y + yoffs[row];
        float xr_[RK];
        if (noisy) {
            if (nm > 1) load_a(rlm[row]);
            if constexpr (RC == 4) {
#pragma unroll
                for (int q = 0; q < RQ; ++q) {
                    const float4 v = *reinterpret_cast<const float4*>(XBs + row * RK + 4 * q);
                    xr_[4 * q] = v.x, xr_[4 * q + 1] = v.y, xr_[4 * q + 2] = v.z, xr_[4 * q + 3] = v.w;
                }
            } else {
                xr_[0] = XBs[row];
            }
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int32_t col = 32 * j + lc;
            if (col >= ct) continue;
            float yv = acc[j][e];
            if (noisy) {
                float z = 0.0f;
#pragma unroll
                for (int c = 0; c < RK; ++c) z = __fadd_rn(z, __fmul_rn(xr_[c], ar[j][c]));
                yv = __fadd_rn(yv, z);
            }
            yrow[col] = yv;
        }
    }
}

static int32_t f32_bn(int32_t a) { return a <= 32 ? 32 : a <= 64 ? 64 : 128; }
static int32_t f32_rk(int32_t r) { return r <= 1 ? 1 : r <= 4 ? 4 : r <= 8 ? 8 : 16; }
static int32_t f32_pad(int32_t a) { return (a + f32_bn(a) - 1) / f32_bn(a) * f32_bn(a); }

// k_gemm_f32s takes do_Tmm (which k_gemm_f32 does not; against k_linear_small, which
// draws a tile's factors in every tile, 1776 rows 64 -> 256 at rank 1 39 -> 13 us, 25600
// rows 64 -> 512 at rank 2 276 -> 54 us) and do_mm with at least 256 outputs over more
// than two K chunks (at b <= 64 such a call is bound by its x and y bytes).  Narrower do_mm outputs are the spiking layers': their currents
// stay on the fp32 chain, because a current at the LIF threshold would spike or
// not with the order of its sum.  The rule is the same for every x format
// (binary inputs give the same bits in all of them).
static bool f32_split_shape(int32_t a, int32_t b, bool tmm) {
    return tmm || (b > 2 * KF_BK && a >= 256);
}
static size_t f32_w_bytes(int32_t a, int32_t b) {
    return (size_t)((b + KF_BK - 1) / KF_BK) * 3 * f32_pad(a) * KF_BK * 2;
}

// Most members a bm-row tile (starting at a multiple of bm) can touch.
static int32_t f32_nm_max(int32_t bm, int32_t R, int32_t n) {
    int32_t nm;
    if (R % bm == 0) nm = 1;
    else if (R > bm) nm = 2;
    else if (bm % R == 0) nm = bm / R;
    else nm = (bm - 1) / R + 2;
    return std::min(nm, n);
}

static int32_t factor_pairs(const LinParams& P) {
    return (int32_t)(((int64_t)P.tid_lo + P.n - 1) / 2 - P.tid_lo / 2 + 1);
}

// Rows per generating thread: up to 16 normals, fewer while that leaves under
// 128k threads (two waves per SIMD); at least enough for the jump tables' row
// count.  1024 pairs x 1024 rows at rank 1: 24.1 us with 64k threads (16 normals
// each), 21.5 with 128k, 33 with 256k (4 normals: the jumps dominate); 2048 x
// 2048: 47 us at 32 normals per thread, 37 at 16, 44 at 8.
static bool factor_rows(const LinParams& P, int32_t* rc_out, int32_t* groups) {
    const int32_t r = P.r, rows = P.a + P.b;
    int32_t rc = std::max(1, 16 / r);
    while (rc > 1 && (int64_t)factor_pairs(P) * ((rows + rc - 1) / rc) < 131072) rc = std::max(1, rc / 2);
    rc = std::max<int32_t>(rc, (int32_t)((rows + kJumpMaxRows - 1) / kJumpMaxRows));
    if ((int64_t)rc * r > kJumpMaxL) return false;
    *rc_out = rc;
    *groups = (rows + rc - 1) / rc;
    return true;
}

// The tiling of one call (shape only).  split: k_gemm_f32s.
struct F32Plan {
    bool split;
    int32_t bm, bn, rk, bch, nm;
    size_t lds, f_bytes, w_bytes;
};

static bool f32_plan(const LinParams& P, bool split, F32Plan* pl) {
    if (P.math != HSES_MATH_F32 || P.r > KF_RMAX || P.r < 0) return false;
    if (split ? !f32_split_shape(P.a, P.b, P.tmm) : P.tmm) return false;
    const int32_t r = P.r;
    pl->split = split;
    pl->bn = f32_bn(P.a);
    pl->bm = KF_BM;
    // split: 64 x 64 tiles while 128-row tiles would leave CUs without one (256 CUs)
    if (split && pl->bn >= 64 && (P.total + 127) / 128 * (f32_pad(P.a) / pl->bn) < 256)
        pl->bm = pl->bn = 64;
    pl->rk = f32_rk(r);
    const int32_t nm = f32_nm_max(pl->bm, P.R, P.n);
    const size_t bch = r > 0 ? (size_t)nm * KF_BK * pl->rk : 0;
    if (bch > (size_t)(split ? KS_BPT : 8) * KF_THREADS) return false;  // BPT values per thread
    pl->bch = (int32_t)bch;
    pl->nm = nm;
    const size_t a_lds = r > 0 ? (size_t)nm * pl->bn * pl->rk : 0;
    if (a_lds > KF_AMAX) return false;
    if (split) {
        const size_t parts = P.x_fmt == HSES_FMT_F32 ? 3 : P.x_fmt == HSES_FMT_BF16 ? 1 : 0;
        pl->lds = (parts * pl->bm + 3 * pl->bn) * KF_BK * 2 + bch * 4 + (size_t)pl->bm * 20 + a_lds * 4;
    } else {
        const size_t nbuf = P.b > KF_BK ? 2 : 1;  // staging buffers (k_gemm_f32)
        pl->lds = (nbuf * ((size_t)(KF_BM + pl->bn) * KF_XP + bch) + a_lds + 3 * KF_BM) * 4;
    }
    pl->w_bytes = split ? f32_w_bytes(P.a, P.b) : 0;
    pl->f_bytes = 0;
    if (r > 0) {
        int32_t rc, groups;
        if (!factor_rows(P, &rc, &groups)) return false;
        pl->f_bytes = align16((size_t)P.n * (P.a + P.b) * r * 4);
    }
    return true;
}

// k_factors: the factor rows (rank 0: none) into F, the split of W into Wp (or NULL).
static int launch_factors_w(LinParams& P, DeviceState* st, hipStream_t s, float* F, uint16_t* Wp,
                            uint16_t* Fb = nullptr) {
    int32_t rc = 1, groups = 0;
    if (P.r > 0) {
        if (!factor_rows(P, &rc, &groups)) return HSES_ERR_UNSUPPORTED;
        int e = get_jump_table(st, (int64_t)rc * P.r, groups, &P.jump);
        if (e) return e;
    }
    const int32_t pairs = factor_pairs(P);
    const int32_t vec = reinterpret_cast<uintptr_t>(F) % 16 == 0 && (int64_t)(P.a + P.b) * P.r % 4 == 0 &&
                        rc * P.r % 4 == 0;
    const int64_t fblocks = ((int64_t)pairs * groups + 255) / 256;
    const int64_t pieces = Wp ? (int64_t)((P.b + KF_BK - 1) / KF_BK) * f32_pad(P.a) * 4 : 0;
    const int64_t blocks = fblocks + (pieces + 255) / 256;
    if (blocks > INT32_MAX) return set_error(HSES_ERR_INVALID_ARG, "too many factor rows");
    hipLaunchKernelGGL(k_factors, dim3((uint32_t)blocks), dim3(256), 0, s, P, rc, groups,
                       pairs, F, Fb, vec, (int32_t)fblocks, Wp, f32_pad(P.a));
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

int launch_factors(LinParams& P, DeviceState* st, hipStream_t s, float* F, uint16_t* Fb) {
    return P.r < 1 ? HSES_ERR_UNSUPPORTED : launch_factors_w(P, st, s, F, nullptr, Fb);
}

size_t linear_f32_workspace(int32_t a, int32_t b, int32_t r, int32_t n, int32_t rows_per_member,
                            int32_t n_time, int32_t math) {
    (void)rows_per_member;
    (void)n_time;
    if (math != HSES_MATH_F32 || a < 1 || b < 1 || n < 1 || r < 0 || r > KF_RMAX) return 0;
    return align16((size_t)n * (a + b) * r * 4) + f32_w_bytes(a, b);
}

template <typename Kern, typename... Args>
static int launch_f32(Kern kern, size_t lds, dim3 grid, hipStream_t s, Args... args) {
    if (lds > 64 * 1024)
        HSES_CHECK_HIP(hipFuncSetAttribute((const void*)kern,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, grid, dim3(KF_THREADS), lds, s, args...);
    HSES_CHECK_HIP(hipGetLastError());
    return HSES_OK;
}

template <int XFMT, int NT>
static int launch_gemm_rk(const LinParams& P, const F32Plan& pl, hipStream_t s, const float* F,
                          dim3 grid) {
    switch (pl.rk) {
        case 1: return launch_f32(k_gemm_f32<XFMT, NT, 1>, pl.lds, grid, s, P, F, pl.bch, pl.nm);
        case 4: return launch_f32(k_gemm_f32<XFMT, NT, 4>, pl.lds, grid, s, P, F, pl.bch, pl.nm);
        case 8: return launch_f32(k_gemm_f32<XFMT, NT, 8>, pl.lds, grid, s, P, F, pl.bch, pl.nm);
        default: return launch_f32(k_gemm_f32<XFMT, NT, 16>, pl.lds, grid, s, P, F, pl.bch, pl.nm);
    }
}

template <int XFMT>
static int launch_gemm_bn(const LinParams& P, const F32Plan& pl, hipStream_t s, const float* F,
                          dim3 grid) {
    switch (pl.bn) {
        case 32: return launch_gemm_rk<XFMT, 1>(P, pl, s, F, grid);
        case 64: return launch_gemm_rk<XFMT, 2>(P, pl, s, F, grid);
        default: return launch_gemm_rk<XFMT, 4>(P, pl, s, F, grid);
    }
}

template <int XFMT, int BM, int BN>
static int launch_split_rk(const LinParams& P, const F32Plan& pl, hipStream_t s, const float* F,
                           const uint16_t* Wp, dim3 grid) {
    const int32_t ap = f32_pad(P.a);
    switch (pl.rk) {
        case 1: return launch_f32(k_gemm_f32s<XFMT, BM, BN, 1>, pl.lds, grid, s, P, F, Wp, ap, pl.bch);
        case 4: return launch_f32(k_gemm_f32s<XFMT, BM, BN, 4>, pl.lds, grid, s, P, F, Wp, ap, pl.bch);
        case 8: return launch_f32(k_gemm_f32s<XFMT, BM, BN, 8>, pl.lds, grid, s, P, F, Wp, ap, pl.bch);
        default: return launch_f32(k_gemm_f32s<XFMT, BM, BN, 16>, pl.lds, grid, s, P, F, Wp, ap, pl.bch);
    }
}

template <int XFMT>
static int launch_split_bn(const LinParams& P, const F32Plan& pl, hipStream_t s, const float* F,
                           const uint16_t* Wp, dim3 grid) {
    if (pl.bm == 64) return launch_split_rk<XFMT, 64, 64>(P, pl, s, F, Wp, grid);
    switch (pl.bn) {
        case 32: return launch_split_rk<XFMT, 128, 32>(P, pl, s, F, Wp, grid);
        case 64: return launch_split_rk<XFMT, 128, 64>(P, pl, s, F, Wp, grid);
        default: return launch_split_rk<XFMT, 128, 128>(P, pl, s, F, Wp, grid);
    }
}

int launch_linear_f32(LinParams& P, DeviceState* st, hipStream_t s, void* work, size_t work_bytes) {
    F32Plan pl;
    auto fits = [&](bool split) {
        return f32_plan(P, split, &pl) && pl.lds <= st->max_lds &&
               (pl.f_bytes + pl.w_bytes == 0 || (work && work_bytes >= pl.f_bytes + pl.w_bytes)) &&
               (!split || reinterpret_cast<uintptr_t>(work) % 16 == 0);
    };
    if (!fits(true) && !fits(false)) return HSES_ERR_UNSUPPORTED;
    const int64_t tiles = (P.total + pl.bm - 1) / pl.bm * ((P.a + pl.bn - 1) / pl.bn);
    if (tiles > INT32_MAX) return set_error(HSES_ERR_INVALID_ARG, "too many output rows");
    float* F = static_cast<float*>(work);
    uint16_t* Wp = pl.split ? reinterpret_cast<uint16_t*>(static_cast<char*>(work) + pl.f_bytes) : nullptr;
    if (P.r > 0 || Wp) {
        const int rc = launch_factors_w(P, st, s, F, Wp);
        if (rc) return rc;
    }
    const dim3 grid((uint32_t)tiles);
    if (pl.split) switch (P.x_fmt) {
        case HSES_FMT_BITS: return launch_split_bn<HSES_FMT_BITS>(P, pl, s, F, Wp, grid);
        case HSES_FMT_BF16: return launch_split_bn<HSES_FMT_BF16>(P, pl, s, F, Wp, grid);
        default: return launch_split_bn<HSES_FMT_F32>(P, pl, s, F, Wp, grid);
    }
    switch (P.x_fmt) {
        case HSES_FMT_BITS: return launch_gemm_bn<HSES_FMT_BITS>(P, pl, s, F, grid);
        case HSES_FMT_BF16: return launch_gemm_bn<HSES_FMT_BF16>(P, pl, s, F, grid);
        default: return launch_gemm_bn<HSES_FMT_F32>(P, pl, s, F, grid);
    }
}

}  // namespace hses
