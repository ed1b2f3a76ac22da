"""The one-launch forward of a few rows (k_linear_few: at most 64 rows) against
float64 of the operands as the kernel takes them.

Bound: in bf16 math products are exact in the fp32 accumulator; in fp32 math each
product and sum of the chains (K / 8 terms per wave, eight waves) rounds, so
rounding errors grow like sqrt(K): 2^-24 (2 sqrt(K) + 16) of the sum of |terms|,
and half a bf16 ulp of a bf16 output."""
import numpy as np
import pytest
import torch

from hyperscalees_amd._lib import FMT_BF16, FMT_BITS, FMT_F32, MATH_BF16, MATH_F32
from tests.test_gpu_linear import KEY, bf16_round, factors, pack_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("math", [MATH_F32, MATH_BF16])
@pytest.mark.parametrize("n,rpm,T,out,inp,r,tid_lo,tmm,fmt", [
    (1, 1, 1, 256, 72, 0, 0, 0, FMT_F32),        # one row, no noise, a ragged K step
    (8, 1, 1, 512, 512, 1, 0, 0, FMT_BF16),      # decoding, one token per member
    (5, 3, 1, 300, 264, 1, 3, 0, FMT_F32),       # odd first member, ragged outputs
    (2, 5, 4, 257, 128, 2, 1, 0, FMT_BF16),      # time-major planes
    (64, 1, 1, 256, 80, 1, 0, 0, FMT_F32),       # the most rows and members
    (3, 21, 1, 17, 104, 4, 2, 1, FMT_F32),       # do_Tmm, narrow
    (16, 2, 1, 40, 256, 1, 1, 1, FMT_BF16),
    (4, 4, 1, 512, 2048, 2, 0, 1, FMT_F32),      # eight K steps per wave
])
def test_few_rows(hses_gpu, n, rpm, T, out, inp, r, tid_lo, tmm, fmt, math):
    rng = np.random.default_rng(out + inp + n)
    rnd = bf16_round if math == MATH_BF16 else (lambda v: v)
    x3 = rng.standard_normal((T, n * rpm, inp)).astype(np.float32)
    xt = torch.from_numpy(x3).cuda()
    if fmt == FMT_BF16:
        xt = xt.to(torch.bfloat16)
        x3 = bf16_round(x3)
    shape = (inp, out) if tmm else (out, inp)
    W = (rng.standard_normal(shape) / np.sqrt(inp)).astype(np.float32)
    Wd, x64 = rnd(W.T if tmm else W).astype(np.float64), rnd(x3).astype(np.float64)
    y, s = x64 @ Wd.T, np.abs(x64) @ np.abs(Wd).T
    if r:
        A, B = factors(0.5, r, n, tid_lo, *shape)
        for m in range(n):
            i, o = (rnd(A[m]), B[m]) if tmm else (rnd(B[m]), A[m])
            rows = slice(m * rpm, (m + 1) * rpm)
            y[:, rows] += (x64[:, rows] @ i.astype(np.float64)) @ o.astype(np.float64).T
            s[:, rows] += (np.abs(x64[:, rows]) @ np.abs(i)) @ np.abs(o).T
    f = hses_gpu.perturbed_linear_t if tmm else hses_gpu.perturbed_linear
    got = f(xt, torch.from_numpy(W).cuda(), KEY, r, 0.5 if r else 0.0, 0, 0, tid_lo, n, rpm, x_fmt=fmt,
            n_time=T, math=math).cpu().numpy().reshape(y.shape)
    tol = 2.0 ** -24 * (2 * np.sqrt(inp) + 16) * s
    assert (np.abs(got - y) <= tol).all(), (np.abs(got - y) / tol).max()


@pytest.mark.parametrize("math", [MATH_F32, MATH_BF16])
@pytest.mark.parametrize("n,rpm,T,out,inp,r,tid_lo,tmm", [
    (2, 16, 1, 256, 784, 4, 0, 0),     # a layer of a few spike rows
    (3, 5, 4, 300, 72, 1, 1, 0),       # ragged outputs, a word's first byte, time-major planes
    (8, 8, 1, 40, 200, 2, 0, 1),       # do_Tmm
    (4, 16, 1, 100, 136, 2, 3, 0),     # narrower outputs
])
def test_few_rows_formats_agree(hses_gpu, n, rpm, T, out, inp, r, tid_lo, tmm, math):
    """Binary inputs give the same bits in every format, whatever lies past a
    packed row's last column."""
    rng = np.random.default_rng(out)
    x3 = (rng.random((T, n * rpm, inp)) < 0.3).astype(np.float32)
    xt = torch.from_numpy(x3).cuda()
    past = np.ones((T, n * rpm, (inp + 63) // 64 * 64), np.float32)
    past[..., :inp] = x3
    shape = (inp, out) if tmm else (out, inp)
    W = torch.from_numpy((rng.standard_normal(shape) / np.sqrt(inp)).astype(np.float32)).cuda()
    f = hses_gpu.perturbed_linear_t if tmm else hses_gpu.perturbed_linear
    ys = [f(x, W, KEY, r, 0.2, 0, 0, tid_lo, n, rpm, x_fmt=fmt, n_time=T, math=math).cpu().numpy()
          for fmt, x in ((FMT_F32, xt), (FMT_BF16, xt.to(torch.bfloat16)), (FMT_BITS, pack_bits(x3)),
                         (FMT_BITS, pack_bits(past)))]
    for y in ys[1:]:
        np.testing.assert_array_equal(ys[0], y)


@pytest.mark.parametrize("act,f", [(1, np.tanh), (2, lambda v: 1 / (1 + np.exp(-v))),
                                   (3, lambda v: np.maximum(v, 0) ** 2)])
def test_few_rows_activation_and_bf16_output(hses_gpu, act, f):
    rng = np.random.default_rng(act)
    x = bf16_round(rng.standard_normal((7, 96)).astype(np.float32))
    W = (rng.standard_normal((96, 33)) / 10).astype(np.float32)
    got = hses_gpu.perturbed_linear_t(torch.from_numpy(x).cuda().to(torch.bfloat16), torch.from_numpy(W).cuda(),
                                      KEY, 1, 0.0, 0, 0, 0, 7, 1, x_fmt=FMT_BF16, math=MATH_BF16, act=act,
                                      out_bf16=True).float().cpu().numpy().reshape(7, 33)
    want = f(x.astype(np.float64) @ bf16_round(W).astype(np.float64))
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 1e-6).all()
