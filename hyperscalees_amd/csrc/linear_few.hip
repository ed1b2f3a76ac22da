// linear_few.hip -- the perturbed forward of a few rows (decoding: one or a few
// tokens of a few members):
//   do_mm  (eggroll.rs:419-446):  y = x W^T + (x B_m) A_m^T,
//   do_Tmm (eggroll.rs:450-477):  y = x W + (x A_m) B_m^T,
// with an optional activation and an fp32 or bf16 output, in one launch.
//
// At a few rows a layer reads W once and computes next to nothing, so its time is
// launches and latency: the wide kernels took three launches (W to bf16, the factor
// draw, a product of one row tile whose K loop is a chain of load latencies), 35 us
// for 8 rows of a 512 x 512 layer.  Here a workgroup of 8 waves owns 16 outputs and
// all rows: every wave loads its share of W (K steps of 32 dealt to the waves in
// turn) straight to registers in the MFMA operand layout, in fp32 as it is stored,
// and while the loads are in flight the workgroup draws the members' input-side
// factors and its 16 output-side rows into LDS (each workgroup again: the draw of
// n b r / 2 normals costs less than a launch and the vector units are idle).  The
// waves' partial sums meet in LDS; 16 outputs per workgroup because more would
// leave CUs without work (a = 512: 32 workgroups) and fewer would repeat the draw.
// 8 rows of 512 x 512 at rank 1, bf16: 15 us (8 without noise), a 512 -> 2048 layer 16,
// an RWKV-7 decode step of 8 members 2.4 -> 1.1 ms of kernels.  The draw and the load
// latencies bound it: two table jumps, four normals and three rounds of L2 loads.
#include <math.h>

#include <type_traits>

#include "linear_common.h"
#include "mfma.h"
#include "noise_dev.h"
#include "runtime.h"

namespace hses {

constexpr int FW_THREADS = 512, FW_WAVES = 8, FW_O = 16, FW_ROWS = 64, FW_BK = 32;
constexpr int FW_NORMALS = 16384;  // input-side normals of all pairs kept in LDS (64 KB)
constexpr int FW_NR = 64;          // members x rank

__device__ __forceinline__ float few_act(float v, int32_t act) {
    if (act == ACT_TANH) return tanhf(v);
    if (act == ACT_SIGMOID) return 1.0f / (1.0f + expf(-v));
    if (act == ACT_RELU_SQ) {
        const float z = v > 0.0f ? v : 0.0f;
        return z * z;
    }
    return v;
}

// 8 consecutive values from p[0], p[st], ... (n of them; zero past n); vec: 16-byte loads
__device__ __forceinline__ void few_load8(const float* p, int64_t st, int32_t n, bool vec, float (&v)[8]) {
    if (vec && n >= 8) {
        const f32x4 a = reinterpret_cast<const f32x4*>(p)[0], b = reinterpret_cast<const f32x4*>(p)[1];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = a[i], v[4 + i] = b[i];
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = i < n ? p[i * st] : 0.0f;
    }
}

__device__ __forceinline__ void few_load8(const uint16_t* p, int32_t n, bool vec, float (&v)[8]) {
    if (vec && n >= 8) {
        const u16x8 u = *reinterpret_cast<const u16x8*>(p);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = bf2f(u[i]);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = i < n ? bf2f(p[i]) : 0.0f;
    }
}

// the 8 bits of a packed row from column k on (n of them), as 0.0 / 1.0
__device__ __forceinline__ void few_load8(const uint64_t* row, int32_t k, int32_t n, float (&v)[8]) {
    uint32_t byte = 0;
    if (n > 0) {
        byte = (uint32_t)(row[k >> 6] >> (k & 63)) & 0xffu;
        if (n < 8) byte &= (1u << n) - 1u;  // bits past the last column may be set
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (float)((byte >> i) & 1u);
}

__device__ __forceinline__ u16x8 few_bf16(const float (&v)[8]) {
    return __builtin_bit_cast(u16x8, uint4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                           pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])});
}

struct FewArgs {
    int32_t pairs, rc;     // pairs of the members; stream rows per drawing item
    int32_t act, ybf16, xvec, wvec;
};

// G: 16-row groups.
template <int MATH, int XFMT, int G>
__global__ __launch_bounds__(FW_THREADS) void k_linear_few(LinParams P, FewArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int32_t a = P.a, b = P.b, r = P.r;
    const int32_t rows = (int32_t)P.total, o0 = blockIdx.x * FW_O, ct = min(FW_O, a - o0);
    // input-side normals [pair][k][r], output-side [pair][16][r], x B_m [row][r],
    // partial sums [wave][row][16], row offsets of y and x, members
    float* Bs = reinterpret_cast<float*>(smem);
    float* Os = Bs + ((size_t)A.pairs * b * r + 3) / 4 * 4;
    float* XB = Os + (size_t)A.pairs * FW_O * r;
    float* Ps = XB + FW_ROWS * r;
    int64_t* yo = reinterpret_cast<int64_t*>(Ps + FW_WAVES * 16 * G * FW_O);
    int64_t* xo = yo + FW_ROWS;
    int32_t* rm = reinterpret_cast<int32_t*>(xo + FW_ROWS);
    BmTables* tabs = reinterpret_cast<BmTables*>(rm + FW_ROWS);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int li = lane & 15, kg = lane >> 4;
    const TileRows tr(P, 0);
    if (tid < rows) {
        yo[tid] = tr.offset(P, tid, P.y_stride, P.y_plane) + o0;
        xo[tid] = tr.offset(P, tid, P.x_stride, P.x_plane);
        rm[tid] = tr.member(P, tid);
    }

    // ---- W of this wave's K steps -------------------------------------------------
    const int32_t steps = (b + FW_BK - 1) / FW_BK;
    const int32_t o = min(o0 + li, a - 1);  // lanes past the tile load its last row, never stored
    auto load_w = [&](int32_t st, float (&w)[8]) {
        const int32_t k = st * FW_BK + 8 * kg, n = min(8, b - k);
        if (P.tmm) few_load8(P.W + (int64_t)k * a + o, a, n, false, w);
        else few_load8(P.W + (int64_t)o * b + k, 1, n, A.wvec, w);
    };
    float w0[8], w1[8];
    if (wave < steps) load_w(wave, w0);
    if (wave + FW_WAVES < steps) load_w(wave + FW_WAVES, w1);

    // ---- the factors -----------------------------------------------------------------
    const int32_t f0 = P.tmm ? a : 0, s0 = (P.tmm ? 0 : b) + o0;  // first input / output side stream row
    if (r > 0) {
        load_bm_tables(tabs, P.tables);
        __syncthreads();
        const NoiseCtx ctx{tabs, P.log_exc, P.cos_exc};
        const int32_t rc = A.rc;
        const int32_t qF0 = f0 / rc, nF = (f0 + b + rc - 1) / rc - qF0;
        const int32_t qS0 = s0 / rc, nS = (s0 + ct + rc - 1) / rc - qS0;
        for (int32_t item = tid; item < A.pairs * (nF + nS); item += FW_THREADS) {
            const int32_t p = item / (nF + nS), qi = item - p * (nF + nS);
            const bool in = qi < nF;
            const int32_t q = in ? qF0 + qi : qS0 + (qi - nF);
            float sign;
            const uint64_t seed = member_seed(P.key, P.epoch, P.nreuse, 2 * (P.tid_lo / 2 + p), &sign);
            uint64_t s = row_start_state(seed, q, P.jump);
            // even members' values (the scaled side times sigma / sqrt(r)); odd ones negate them
            const float sc = in == (P.tmm != 0) ? P.bs : 1.0f;
            const int32_t first = in ? f0 : s0, cnt = in ? b : ct;
            float* dst = in ? Bs + (size_t)p * b * r : Os + (size_t)p * FW_O * r;
            bm_run(s, min(rc, a + b - q * rc) * r, ctx, [&](int32_t i, float v) {
                const int32_t e = (q * rc - first) * r + i;  // a group may start before the range
                if (e >= 0 && e < cnt * r) dst[e] = v * sc;
            });
        }
    }
    __syncthreads();
    // x B_m: a wave per row, lanes over k
    auto pair_of = [&](int32_t m) { return (P.tid_lo + m) / 2 - P.tid_lo / 2; };
    if (r > 0) {
        for (int32_t row = wave; row < rows; row += FW_WAVES) {
            const int32_t m = rm[row];
            const float* bs = Bs + (size_t)pair_of(m) * b * r;
            const bool neg = P.tmm && ((P.tid_lo + m) & 1);
            for (int32_t c = 0; c < r; ++c) {
                float z = 0.0f;
                for (int32_t k = lane; k < b; k += 64) {
                    float x;
                    if constexpr (XFMT == HSES_FMT_F32) x = static_cast<const float*>(P.x)[xo[row] + k];
                    else if constexpr (XFMT == HSES_FMT_BF16) x = bf2f(static_cast<const uint16_t*>(P.x)[xo[row] + k]);
                    else x = (float)((static_cast<const uint64_t*>(P.x)[xo[row] + (k >> 6)] >> (k & 63)) & 1u);
                    float f = bs[(size_t)k * r + c];
                    if constexpr (MATH == HSES_MATH_BF16) {
                        x = bf2f(f2bf(x));
                        f = bf2f(f2bf(f));
                    }
                    z = __builtin_fmaf(x, f, z);
                }
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) z += __shfl_xor(z, d);
                if (lane == 0) XB[row * r + c] = neg ? -z : z;
            }
        }
    }

    // ---- x W^T: D[output][row] of this wave's K steps --------------------------------
    f32x4 acc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = f32x4{0, 0, 0, 0};
    int64_t xoff[G];
#pragma unroll
    for (int g = 0; g < G; ++g) xoff[g] = xo[min(16 * g + li, rows - 1)];
    auto step = [&](int32_t st, const float (&w)[8]) {
        const int32_t k = st * FW_BK + 8 * kg, n = min(8, b - k);
        u16x8 wb;
        if constexpr (MATH == HSES_MATH_BF16) wb = few_bf16(w);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float x[8];
            if constexpr (XFMT == HSES_FMT_F32)
                few_load8(static_cast<const float*>(P.x) + xoff[g] + k, 1, n, A.xvec, x);
            else if constexpr (XFMT == HSES_FMT_BF16)
                few_load8(static_cast<const uint16_t*>(P.x) + xoff[g] + k, n, A.xvec, x);
            else
                few_load8(static_cast<const uint64_t*>(P.x) + xoff[g], k, n, x);
            if constexpr (MATH == HSES_MATH_BF16) {
                acc[g] = mfma_bf16(wb, few_bf16(x), acc[g]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[g] = mfma_f32(w[i], x[i], acc[g]);
            }
        }
    };
    for (int32_t st = wave; st < steps; st += 2 * FW_WAVES) {
        step(st, w0);
        if (st + 2 * FW_WAVES < steps) load_w(st + 2 * FW_WAVES, w0);
        if (st + FW_WAVES < steps) step(st + FW_WAVES, w1);
        if (st + 3 * FW_WAVES < steps) load_w(st + 3 * FW_WAVES, w1);
    }
    // lane (li, kg): outputs 4 kg .. + 4 of row 16 g + li
#pragma unroll
    for (int g = 0; g < G; ++g)
        *reinterpret_cast<f32x4*>(Ps + ((size_t)wave * 16 * G + 16 * g + li) * FW_O + 4 * kg) = acc[g];
    __syncthreads();

    // ---- the waves' sums in wave order, the rank-r term, the activation -------------------
    for (int32_t e = tid; e < rows * FW_O; e += FW_THREADS) {
        const int32_t row = e / FW_O, c0 = e % FW_O;
        if (c0 >= ct) continue;
        float y = 0.0f;
#pragma unroll
        for (int w = 0; w < FW_WAVES; ++w) y += Ps[((size_t)w * 16 * G + row) * FW_O + c0];
        if (r > 0) {
            const int32_t m = rm[row];
            const float* os = Os + ((size_t)pair_of(m) * FW_O + c0) * r;
            const bool neg = !P.tmm && ((P.tid_lo + m) & 1);
            float z = 0.0f;
            for (int32_t c = 0; c < r; ++c) z = __fadd_rn(z, __fmul_rn(XB[row * r + c], neg ? -os[c] : os[c]));
            y = __fadd_rn(y, z);
        }
        y = few_act(y, A.act);
        if (A.ybf16) reinterpret_cast<uint16_t*>(P.y)[yo[row] + c0] = f2bf(y);
        else P.y[yo[row] + c0] = y;
    }
}

// Few enough rows that one tile holds them, few enough members and normals that
// every workgroup can draw them, within the shapes the tiled small-rank kernels
// take (members x rank <= 64 per tile).  fp32 math: the layers k_gemm_f32s takes
// (narrower ones stay on their fp32 chains, see f32_split_shape).  The rule is the
// same for every x format: binary inputs give the same bits in all of them.
int launch_linear_few(LinParams& P, DeviceState* st, hipStream_t s, int32_t act, int32_t y_fmt) {
    if (P.total > FW_ROWS) return HSES_ERR_UNSUPPORTED;
    const bool bf = P.math == HSES_MATH_BF16;
    if (!bf && (P.b <= 64 || !(P.tmm || P.a >= 256) || y_fmt != HSES_FMT_F32)) return HSES_ERR_UNSUPPORTED;
    LinParams Q = P;
    Q.r = (P.r > 0 && P.bs != 0.0f) ? P.r : 0;
    FewArgs A{};
    A.pairs = Q.r > 0 ? (int32_t)(((int64_t)P.tid_lo + P.n - 1) / 2 - P.tid_lo / 2 + 1) : 0;
    if ((int64_t)P.n * Q.r > FW_NR || (int64_t)A.pairs * P.b * Q.r > FW_NORMALS) return HSES_ERR_UNSUPPORTED;
    A.act = act;
    A.ybf16 = y_fmt == HSES_FMT_BF16;
    const int64_t vec = P.x_fmt == HSES_FMT_F32 ? 4 : 8;
    A.xvec = reinterpret_cast<uintptr_t>(P.x) % 16 == 0 && P.x_stride % vec == 0 &&
             (P.n_time == 1 || P.x_plane % vec == 0);
    A.wvec = reinterpret_cast<uintptr_t>(P.W) % 16 == 0 && P.b % 4 == 0;
    A.rc = 1;
    if (Q.r > 0) {
        // rows per drawing item: one round of items where the jump table allows it
        const int32_t rows = P.a + P.b;
        while (A.rc < 16 && (int64_t)A.pairs * (P.b / A.rc) > FW_THREADS && 2 * A.rc * Q.r <= 16) A.rc *= 2;
        const int rc = get_jump_table(st, (int64_t)A.rc * Q.r, (rows + A.rc - 1) / A.rc, &Q.jump);
        if (rc) return rc;
    }
    auto launch = [&](auto kern, int g) -> int {
        const size_t lds = (((size_t)A.pairs * P.b * Q.r + 3) / 4 * 4 + (size_t)A.pairs * FW_O * Q.r +
                            FW_ROWS * Q.r + (size_t)FW_WAVES * 16 * g * FW_O) * 4 +
                           FW_ROWS * 20 + (Q.r > 0 ? sizeof(BmTables) : 0);
        if (lds > st->max_lds) return HSES_ERR_UNSUPPORTED;
        if (lds > 64 * 1024)
            HSES_CHECK_HIP(hipFuncSetAttribute((const void*)kern,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kern, dim3((P.a + FW_O - 1) / FW_O), dim3(FW_THREADS), lds, s, Q, A);
        HSES_CHECK_HIP(hipGetLastError());
        return HSES_OK;
    };
    auto by_g = [&](auto mc, auto xc) -> int {
        constexpr int M = decltype(mc)::value, X = decltype(xc)::value;
        if (P.total <= 16) return launch(k_linear_few<M, X, 1>, 1);
        if (P.total <= 32) return launch(k_linear_few<M, X, 2>, 2);
        return launch(k_linear_few<M, X, 4>, 4);
    };
    using std::integral_constant;
    auto by_x = [&](auto mc) -> int {
        return P.x_fmt == HSES_FMT_F32    ? by_g(mc, integral_constant<int, HSES_FMT_F32>{})
               : P.x_fmt == HSES_FMT_BF16 ? by_g(mc, integral_constant<int, HSES_FMT_BF16>{})
                                          : by_g(mc, integral_constant<int, HSES_FMT_BITS>{});
    };
    return bf ? by_x(integral_constant<int, HSES_MATH_BF16>{}) : by_x(integral_constant<int, HSES_MATH_F32>{});
}

}  // namespace hses
