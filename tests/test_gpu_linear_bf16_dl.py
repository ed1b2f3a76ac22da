"""The bf16 forward with its rank-1 terms on the matrix cores (k_gemm_bf16_dl:
rank 0 or 1, outputs at least 256 wide, inputs a multiple of 32) against
float64 of the operands as the kernel takes them: x, W and the input-side
factor rounded to bf16, the output-side factor in fp32.

Bound: products of bf16 values are exact in the fp32 accumulator; rounding of
the running sums (one per 16 k, random) and of the rank-1 term's, whose parts
leave out less than 2^-25 of it: 2^-24 (2 sqrt(K) + 16) of the sum of |terms|."""
import numpy as np
import pytest
import torch

from hyperscalees_amd._lib import FMT_BF16, FMT_F32, MATH_BF16
from tests.test_gpu_linear import KEY, bf16_round, factors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rpm,T,out,inp,r,tid_lo,tmm,fmt", [
    (1, 1, 1, 256, 32, 1, 0, 0, FMT_BF16),       # one row, one step
    (7, 43, 1, 260, 64, 1, 1, 0, FMT_BF16),      # four members in a tile, odd first, ragged columns
    (3, 129, 1, 512, 96, 1, 0, 0, FMT_F32),      # three steps, rows past a tile
    (2, 200, 3, 256, 160, 1, 0, 0, FMT_BF16),    # time-major planes
    (5, 64, 1, 768, 2048, 1, 2, 0, FMT_F32),     # two members per tile, 64 steps
    (4, 100, 1, 300, 128, 1, 1, 1, FMT_BF16),    # do_Tmm
    (4, 100, 1, 512, 128, 0, 0, 1, FMT_F32),     # no noise
])
@pytest.mark.parametrize("act", [0, 3])
def test_rank1_terms_on_matrix_cores(hses_gpu, n, rpm, T, out, inp, r, tid_lo, tmm, fmt, act):
    rng = np.random.default_rng(out + inp + n)
    x3 = bf16_round(rng.standard_normal((T, n * rpm, inp)).astype(np.float32))
    shape = (inp, out) if tmm else (out, inp)
    W = (rng.standard_normal(shape) / np.sqrt(inp)).astype(np.float32)
    Wd = bf16_round(W.T if tmm else W).astype(np.float64)
    x64 = x3.astype(np.float64)
    y, s = x64 @ Wd.T, np.abs(x64) @ np.abs(Wd).T
    if r:
        A, B = factors(0.5, r, n, tid_lo, *shape)
        for m in range(n):
            i, o = (bf16_round(A[m]), B[m]) if tmm else (bf16_round(B[m]), A[m])
            rows = slice(m * rpm, (m + 1) * rpm)
            y[:, rows] += (x64[:, rows] @ i.astype(np.float64)) @ o.astype(np.float64).T
            s[:, rows] += (np.abs(x64[:, rows]) @ np.abs(i)) @ np.abs(o).T
    f = hses_gpu.perturbed_linear_t if tmm else hses_gpu.perturbed_linear
    xt = torch.from_numpy(x3).cuda()
    xt = xt.to(torch.bfloat16) if fmt == FMT_BF16 else xt
    out_bf = act == 3
    got = f(xt, torch.from_numpy(W).cuda(), KEY, r, 0.5 if r else 0.0, 0, 0, tid_lo, n, rpm, x_fmt=fmt,
            n_time=T, math=MATH_BF16, act=act, out_bf16=out_bf)
    got = got.float().cpu().numpy().reshape(y.shape)
    tol = 2.0 ** -24 * (2 * np.sqrt(inp) + 16) * s
    if act == 3:   # relu(y)^2 moves by (|y| + tol)^2 - y^2, stored as bf16
        tol = tol * (2 * np.abs(y) + tol)
        y = np.maximum(y, 0.0) ** 2
        tol = tol + 2.0 ** -8 * (y + tol)
    assert (np.abs(got - y) <= tol).all(), (np.abs(got - y) / tol).max()


def test_rank1_term_of_infinite_rows(hses_gpu):
    """An infinite x B_m keeps its sign through the rank-1 term: a zero W leaves
    +-inf (NaN where the output-side factor is 0), as an fp32 product does."""
    n, rpm, out, inp = 2, 64, 256, 32
    x = np.zeros((n * rpm, inp), np.float32)
    x[5, 3], x[70, 8] = np.inf, -np.inf
    xt = torch.from_numpy(x).cuda().to(torch.bfloat16)
    W = torch.full((out, inp), 0.5, device="cuda")
    got = hses_gpu.perturbed_linear(xt, W, KEY, 1, 0.5, 0, 0, 0, n, rpm, x_fmt=FMT_BF16,
                                    math=MATH_BF16).cpu().numpy().reshape(n * rpm, out)
    A, B = factors(0.5, 1, n, 0, out, inp)
    with np.errstate(all="ignore"):
        for row, m in ((5, 0), (70, 1)):
            k = 3 if row == 5 else 8
            xb = np.float64(x[row, k]) * B[m][k, 0]
            want = np.float64(x[row, k]) * 0.5 + xb * A[m][:, 0].astype(np.float64)
            # inf - inf is NaN in both; otherwise the same infinity.  (0 x inf of the
            # other columns of W does not arise: x is 0 there and W finite.)
            np.testing.assert_array_equal(np.isnan(got[row]), np.isnan(want))
            np.testing.assert_array_equal(got[row][~np.isnan(want)], want[~np.isnan(want)])
    rest = np.delete(got, [5, 70], 0)
    assert (rest == 0).all()


@pytest.mark.parametrize("n,rpm,tmm", [(1, 128, 0), (5, 43, 0), (5, 43, 1)])
@pytest.mark.parametrize("e", [-118, -60, 40, 127])
def test_rank1_term_past_the_parts_range(hses_gpu, n, rpm, tmm, e):
    """Factors whose third bf16 part is lost (sigma 2^-118) or that reach fp32's largest
    (2^127: some are infinite) give the fp32 product of the two factors, in their own
    member's rows alone.  W is 0, so y is the rank-1 term; x is 0 but for one value a
    row, so x B_m is one product, exact in fp32 or rounded by the scaled side."""
    rng = np.random.default_rng(1000 + n + e)
    out, inp, sigma = 512, 64, 2.0 ** e
    x = np.zeros((n * rpm, inp), np.float32)
    cols = rng.integers(0, inp, n * rpm)
    small = 2.0 ** -20 if e > 0 else 1.0
    x[np.arange(n * rpm), cols] = bf16_round(rng.uniform(0.5, 2.0, n * rpm).astype(np.float32)) * np.float32(small)
    W = torch.zeros((inp, out) if tmm else (out, inp), device="cuda")
    f = hses_gpu.perturbed_linear_t if tmm else hses_gpu.perturbed_linear
    got = f(torch.from_numpy(x).cuda().to(torch.bfloat16), W, KEY, 1, sigma, 0, 0, 1, n, rpm, x_fmt=FMT_BF16,
            math=MATH_BF16).cpu().numpy().reshape(n * rpm, out)
    with np.errstate(all="ignore"):
        A, B = factors(sigma, 1, n, 1, inp, out) if tmm else factors(sigma, 1, n, 1, out, inp)
        for m in range(n):
            rows = slice(m * rpm, (m + 1) * rpm)
            i, o = (bf16_round(A[m]), B[m]) if tmm else (bf16_round(B[m]), A[m])
            xb = (x[rows, :].astype(np.float64) * i[:, 0].astype(np.float64)).sum(1)  # 0 x inf: NaN
            want = xb[:, None] * o[:, 0].astype(np.float64)
            want[np.abs(want) > 3.4028235e38 * (1 + 2.0 ** -24)] *= np.inf
            fin = np.isfinite(want)
            np.testing.assert_array_equal(got[rows][~fin], want[~fin].astype(np.float32))
            # one rounding of the product (of the parts' sums: six) or an ulp of fp32's
            # subnormals; do_Tmm sums small x A_m on the matrix cores, which may take
            # subnormals as 0
            least = 2.0 ** (-126 if tmm else -148)
            assert (np.abs(got[rows] - want)[fin] <= 2.0 ** -21 * np.abs(want[fin]) + least).all()
