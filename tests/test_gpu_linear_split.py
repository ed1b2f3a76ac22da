"""The fp32 forward on split operands (k_gemm_f32s: do_Tmm, and do_mm with at
least 256 outputs over inputs more than 64 wide) against float64.

Bound: a product of two bf16 parts is exact in the fp32 accumulator, the
products left out are below 2^-25 of |x w|, and a running sum is rounded at most
once per k and part product plus the few roundings that put the sums together;
each is at most half an ulp of a partial sum below sum |x w|.  Rounding errors
of K terms grow like sqrt(K): 2^-24 (4 sqrt(K) + 8) of the sum of |terms|."""
import numpy as np
import pytest
import torch

from hyperscalees_amd._lib import FMT_BF16, FMT_BITS, FMT_F32
from tests import oracle_lib as O
from tests.test_gpu_linear import KEY, factors, pack_bits

pytestmark = pytest.mark.gpu


def reference(x3, W, A, B, rpm, tmm):
    """float64 y and sum of |terms|; W is (out, in), or (in, out) for do_Tmm."""
    Wd = (W.T if tmm else W).astype(np.float64)
    y, s = x3 @ Wd.T, np.abs(x3) @ np.abs(Wd).T
    for m in range(A.shape[0] if A is not None else 0):
        i, o = (A[m], B[m]) if tmm else (B[m], A[m])
        rows = slice(m * rpm, (m + 1) * rpm)
        y[:, rows] += (x3[:, rows] @ i.astype(np.float64)) @ o.astype(np.float64).T
        s[:, rows] += (np.abs(x3[:, rows]) @ np.abs(i)) @ np.abs(o).T
    return y, s


@pytest.mark.parametrize("n,rpm,T,out,inp,r,tid_lo,tmm,fmt", [
    (2, 300, 1, 256, 65, 1, 0, 0, FMT_F32),      # shortest split K, a ragged last chunk
    (5, 131, 1, 257, 96, 2, 1, 0, FMT_F32),      # one column past a tile, odd first member
    (3, 37, 3, 1000, 99, 4, 0, 0, FMT_F32),      # unaligned rows, members straddle tiles
    (2, 512, 40, 300, 784, 4, 1, 0, FMT_BITS),   # 128-row tiles, bit-packed
    (40, 257, 1, 384, 160, 8, 0, 0, FMT_BF16),   # 128-row tiles, bf16 x
    (300, 128, 1, 256, 72, 16, 0, 0, FMT_F32),   # largest rank
    (1, 1, 1, 256, 66, 0, 0, 0, FMT_F32),        # one row, no noise
    (4, 50, 1, 10, 100, 4, 3, 1, FMT_F32),       # do_Tmm, 32-column tile
    (70, 500, 1, 33, 130, 1, 0, 1, FMT_F32),     # do_Tmm, 64-column tile, 128 rows
    (9, 40, 2, 70, 256, 1, 1, 1, FMT_BF16),      # do_Tmm, two column tiles
    (6, 64, 2, 130, 200, 2, 0, 1, FMT_BITS),
    (48, 37, 1, 256, 64, 1, 0, 1, FMT_F32),      # do_Tmm over two K chunks
    (5, 50, 1, 300, 20, 4, 1, 1, FMT_F32),       # over part of one
    (3, 100, 2, 17, 1, 1, 0, 1, FMT_BF16),       # over one input
])
def test_split_against_float64(hses_gpu, n, rpm, T, out, inp, r, tid_lo, tmm, fmt):
    rng = np.random.default_rng(out + inp + r)
    x3 = rng.standard_normal((T, n * rpm, inp)).astype(np.float32)
    x3 *= np.exp2(rng.integers(-12, 13, inp)).astype(np.float32)   # no common scale
    if fmt == FMT_BITS:
        x3 = (x3 > 0).astype(np.float32)
        xt = pack_bits(x3)
    elif fmt == FMT_BF16:
        xt = torch.from_numpy(x3).to(torch.bfloat16).cuda()
        x3 = xt.float().cpu().numpy()
    else:
        xt = torch.from_numpy(x3).cuda()
    shape = (inp, out) if tmm else (out, inp)
    W = (rng.standard_normal(shape) / np.sqrt(inp)).astype(np.float32)
    A = B = None
    if r:
        A, B = factors(0.2, r, n, tid_lo, *shape)
    ref, s = reference(x3.astype(np.float64), W, A, B, rpm, tmm)
    f = hses_gpu.perturbed_linear_t if tmm else hses_gpu.perturbed_linear
    y = f(xt, torch.from_numpy(W).cuda(), KEY, r, 0.2 if r else 0.0, 0, 0, tid_lo, n, rpm, x_fmt=fmt,
          n_time=T).cpu().numpy().reshape(ref.shape)
    # x B_m and (x B_m) A_m^T run as fp32 chains of inp and r terms
    tol = 2.0 ** -24 * (4 * np.sqrt(inp + r) + 8)
    err = (np.abs(y - ref) / s).max()
    assert err <= tol, f"error {err:.2e} of the sum of |terms|, bound {tol:.2e}"


@pytest.mark.parametrize("n,inp,out,tmm,fmt,xe,we", [
    (150, 100, 300, 0, FMT_F32, -121, 0),    # x below the parts' range
    (70, 66, 256, 0, FMT_F32, 0, -121),      # W
    (130, 97, 270, 0, FMT_F32, -120, 30),    # x, against large weights
    (90, 64, 40, 1, FMT_F32, -60, -60),      # the part products
    (129, 130, 70, 1, FMT_BF16, 0, -121),
    (200, 80, 260, 0, FMT_BITS, 0, -121),
])
def test_split_small_magnitudes(hses_gpu, n, inp, out, tmm, fmt, xe, we):
    """Operands so small that their bf16 parts lose bits keep the fp32 bar; rows of
    zeros beside them stay zero."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, inp)).astype(np.float32)
    x = (x > 0).astype(np.float32) if fmt == FMT_BITS else x * np.float32(2.0 ** xe)
    x[5] = 0.0
    xt = torch.from_numpy(x).cuda()
    if fmt == FMT_BITS:
        xt = pack_bits(x[None])
    elif fmt == FMT_BF16:
        xt = xt.to(torch.bfloat16)
        x = xt.float().cpu().numpy()
    W = (rng.standard_normal((inp, out) if tmm else (out, inp)) * np.float32(2.0 ** we)).astype(np.float32)
    Wd = (W.T if tmm else W).astype(np.float64)
    f = hses_gpu.perturbed_linear_t if tmm else hses_gpu.perturbed_linear
    y = f(xt, torch.from_numpy(W).cuda(), KEY, 0, 0.0, 0, 0, 0, n, 1, x_fmt=fmt).cpu().numpy().reshape(n, out)
    ref, s = x.astype(np.float64) @ Wd.T, np.abs(x).astype(np.float64) @ np.abs(Wd).T
    err = np.abs(y - ref) / np.maximum(s, 1e-300)
    assert not y[5].any()
    assert err.max() <= 2.0 ** -24 * (4 * np.sqrt(inp) + 8), err.max()


def test_split_values_without_parts(hses_gpu):
    """Infinities, NaN and magnitudes that round up past bf16's range give what an
    fp32 chain gives, and leave the other rows and columns alone."""
    rng = np.random.default_rng(3)
    n, inp, out = 300, 100, 300
    x = rng.standard_normal((n, inp)).astype(np.float32)
    W = rng.standard_normal((out, inp)).astype(np.float32)
    x[3, 7], x[140, 0], x[141, 99], x[200, 5] = np.inf, np.nan, -np.inf, np.float32(3.4e38)
    x[200, :5], x[200, 6:] = 0.0, 0.0
    W[17, 50], W[280, 3], W[:, 5] = np.inf, np.nan, np.clip(W[:, 5], -0.9, 0.9)
    y = hses_gpu.perturbed_linear(torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda(), KEY, 0, 0.0, 0,
                                  0, 0, n, 1).cpu().numpy().reshape(n, out)
    with np.errstate(all="ignore"):
        ref = x.astype(np.float64) @ W.astype(np.float64).T
        s = np.abs(x).astype(np.float64) @ np.abs(W).astype(np.float64).T
    fin = np.isfinite(ref)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(y[~fin & ~np.isnan(ref)], ref[~fin & ~np.isnan(ref)])
    assert (np.abs(y[fin] - ref[fin]) <= 2.0 ** -24 * (4 * np.sqrt(inp) + 8) * s[fin]).all()


@pytest.mark.parametrize("value", [2.0 ** -80, 0.0, np.inf])
def test_split_rows_past_the_range_leave_others_alone(hses_gpu, value):
    """A row of sums below 2^-60, of zeros or of infinities in a tile: the other rows keep
    their bits (only its own outputs are formed again on fp32 chains)."""
    rng = np.random.default_rng(5)
    n, inp, out = 260, 130, 300
    x = torch.from_numpy(rng.standard_normal((n, inp)).astype(np.float32)).cuda()
    W = torch.from_numpy(rng.standard_normal((out, inp)).astype(np.float32)).cuda()

    def run():
        return hses_gpu.perturbed_linear(x.view(1, n, inp), W, KEY, 1, 0.2, 0, 0, 0, n // 4, 4).view(n, out)

    before = run().clone()
    rows = torch.tensor([0, 77, 259], device="cuda")
    x[rows] = x[rows].sign() * value if value < np.inf else value
    after = run()
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[rows] = False
    assert torch.equal(after[keep], before[keep])
    assert not torch.equal(after[rows], before[rows])
