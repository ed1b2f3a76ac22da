"""The ES update's own record (hses_es_update: k_es_draw, then k_es_gemm below
rank 32 or k_es_rows) against the oracle's double-accumulated sum, at the edges of
its tiles, K chunks and pair ranges.

Bound: the split operands leave out less than 2^-20 of a term (2^-24 below rank 32,
where they keep 24 bits) and each of the K
fp32 sums rounds by half an ulp of a partial sum: 2^-20 + 2^-24 sqrt(K) of the sum
of |terms|, which by the normals' independence is below sqrt(K) times the
gradient's root mean square per element."""
import math

import numpy as np
import pytest
import torch

from hyperscalees_amd import _lib
from tests.test_gpu_update import KEY, gpu_grad, oracle_grad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a,b,r,n,tid_lo", [
    (1, 1, 1, 2, 0),            # one pair, one output
    (1, 5, 1, 1, 3),            # one unpaired member
    (129, 127, 1, 33, 1),       # one row past a tile; K chunks that pairs do not fill
    (128, 128, 1, 4096, 0),     # aligned groups of four (wide stores), 32 splits
    (130, 386, 3, 301, 5),      # a chunk ends inside a pair
    (64, 64, 8, 1024, 0),
    (300, 20, 31, 77, 2),       # largest rank of the chunked form
    (200, 500, 48, 301, 0),     # k_es_rows from the record, several tiles
    (10, 33, 32, 40, 1),
])
def test_own_record(hses_gpu, a, b, r, n, tid_lo):
    fit = np.random.default_rng(a + b + r).standard_normal(n).astype(np.float32)
    ref = oracle_grad(0.02, r, fit, a, b, tid_lo)
    g = gpu_grad(hses_gpu, 0.02, r, fit, a, b, np.float32(1.0), tid_lo).cpu().numpy()
    K = (n + 1) // 2 * r + r
    tol = (2.0 ** -20 + 2.0 ** -24 * math.sqrt(K)) * math.sqrt(K) * max(np.sqrt((ref ** 2).mean()),
                                                                        np.abs(ref).max() / 8)
    assert np.abs(g - ref).max() <= tol, (np.abs(g - ref).max(), tol)
    # a second call into the same workspace, and one that adds
    g2 = gpu_grad(hses_gpu, 0.02, r, fit, a, b, np.float32(1.0), tid_lo)
    assert np.array_equal(g, g2.cpu().numpy())
    g3 = gpu_grad(hses_gpu, 0.02, r, fit, a, b, np.float32(1.0), tid_lo, out=g2.clone(), accumulate=True)
    assert torch.equal(g3, g2 + g2)


def test_zero_fitness_and_scale_range(hses_gpu):
    """All-zero fitness gives zeros; fitness at either end of fp32 keeps the
    relative bar (the operands keep fp32's range)."""
    fit = np.zeros(64, np.float32)
    assert not gpu_grad(hses_gpu, 0.1, 2, fit, 40, 50, np.float32(1.0)).any()
    base = np.random.default_rng(1).standard_normal(64).astype(np.float32)
    ref = oracle_grad(0.1, 2, base, 40, 50)
    for e in (-60, 60):
        g = gpu_grad(hses_gpu, 0.1, 2, base * np.float32(2.0 ** e), 40, 50, np.float32(2.0 ** -e))
        assert np.abs(g.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("a,b,r,n,splits", [
    (64, 64, 8, 1024, 64),      # k_es_partial's splits: 512 pairs / 8
    (200, 500, 48, 302, 18),    # k_es_rows': 151 pairs / 8
])
def test_workspace_of_partials_alone(hses_gpu, a, b, r, n, splits):
    """A workspace that holds the partials and the scale but no record draws inside
    the contraction; one too small for the partials is refused."""
    fit = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    ref = oracle_grad(0.02, r, fit, a, b, 0)
    f, g = torch.from_numpy(fit).cuda(), torch.empty((a, b), device="cuda")
    work = torch.empty(splits * a * b * 4 + 16, dtype=torch.uint8, device="cuda")

    def call(nbytes):
        _lib.call("hses_es_update", f.data_ptr(), n, 0, KEY & (2 ** 64 - 1), r, 0.02, 0, 0, a, b, 1.0, 0,
                  g.data_ptr(), work.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)

    call(work.numel())
    K = n // 2 * r
    tol = (2.0 ** -20 + 2.0 ** -24 * math.sqrt(K)) * math.sqrt(K) * max(np.sqrt((ref ** 2).mean()),
                                                                        np.abs(ref).max() / 8)
    assert np.abs(g.cpu().numpy() - ref).max() <= tol
    with pytest.raises(_lib.HsesError):
        call(a * b * 4)


@pytest.mark.parametrize("a,b,n,tid_lo", [(130, 386, 1, 0), (5, 7, 1, 3), (128, 256, 2, 0), (257, 64, 2, 4)])
def test_one_pair_keeps_fp32_operands(hses_gpu, a, b, n, tid_lo):
    """One pair at rank 1: every output is one product of fp32 operands, within the
    roundings of the weight, of the weighted factor and of the product (half an ulp
    each, 2^-24) and 2^-24 for the part products left out, of |term|; the operands'
    zeros aside, small values included."""
    fit = np.random.default_rng(a).standard_normal(n).astype(np.float32)
    ref = oracle_grad(0.02, 1, fit, a, b, tid_lo)
    # odd members carry the even ones' noise negated: their terms add up
    s = np.abs(oracle_grad(0.02, 1, np.abs(fit) * np.where(np.arange(n) % 2, -1.0, 1.0), a, b, tid_lo))
    g = gpu_grad(hses_gpu, 0.02, 1, fit, a, b, np.float32(1.0), tid_lo).cpu().numpy()
    assert (np.abs(g - ref) <= 4 * 2.0 ** -24 * s).all(), (np.abs(g - ref) / s).max()


@pytest.mark.parametrize("a,b,r,n,e", [
    (40, 50, 2, 64, -100), (40, 50, 2, 64, 100),    # 2^e alone is a scale fp32 holds
    (40, 50, 2, 64, -115), (40, 50, 2, 64, 119),    # a scale that is not
    (130, 70, 1, 301, -110), (130, 70, 1, 301, 118),
    (20, 140, 16, 33, -112), (20, 140, 16, 33, 120),
])
def test_fitness_near_the_ends_of_fp32(hses_gpu, a, b, r, n, e):
    """A finite fitness whose terms are near fp32's ends gives the scaled gradient."""
    base = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    ref = oracle_grad(0.1, r, base, a, b)
    g = gpu_grad(hses_gpu, 0.1, r, base * np.float32(2.0 ** e), a, b, np.float32(2.0 ** -e)).cpu().numpy()
    assert np.isfinite(g).all()
    # a fp32 chain of K terms: 2^-24 sqrt(K) of the sum of |terms|, below sqrt(K) times
    # the gradient's root mean square; and three roundings of a term
    K = (n + 1) // 2 * r
    tol = 2.0 ** -24 * (math.sqrt(K) + 4) * math.sqrt(K) * max(np.sqrt((ref ** 2).mean()),
                                                               np.abs(ref).max() / 8)
    assert np.abs(g - ref).max() <= tol, (np.abs(g - ref).max(), tol)


@pytest.mark.parametrize("n,bad", [(64, np.inf), (301, -np.inf), (64, 1.0e38)])
def test_fitness_past_the_operand_halves(hses_gpu, n, bad):
    """One fitness that is infinite, or whose terms reach fp32's range, at rank 1:
    infinities where fp32 chains have them, with their signs, and no NaN."""
    fit = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    fit[5] = bad
    a, b = 130, 200
    g = gpu_grad(hses_gpu, 1.0, 1, fit, a, b, np.float32(1.0)).cpu().numpy()
    lone = np.zeros(n, np.float32)
    lone[5] = np.sign(bad)
    sign = oracle_grad(1.0, 1, lone, a, b)  # member 5's term
    assert not np.isnan(g).any() and (np.abs(sign) > 0).all()
    if np.isinf(bad):
        assert np.array_equal(g, np.sign(sign) * np.float32(np.inf))
    else:
        big = np.abs(sign) > 1e-3  # against which the other members' terms vanish
        ref = sign * 1.0e38       # its A operands stay below fp32's largest
        safe = big & (np.abs(ref) < 3.3e38)
        over = np.abs(ref) > 3.5e38
        assert safe.any() and over.any()
        assert np.allclose(g[safe], ref[safe], rtol=2.0 ** -21)  # three roundings
        assert np.array_equal(g[over], np.sign(sign[over]) * np.float32(np.inf))


@pytest.mark.parametrize("a,b,r,n", [
    (24, 200, 4, 320_000),    # 256 splits: the last 19 add to the first 19 partials
    (2048, 4096, 1, 90_001),  # one split a part, three parts; the last pair is one member
])
def test_record_in_parts(hses_gpu, a, b, r, n):
    """A record past its bound (512 MB) runs in parts that add to the same partials.
    Against the sum of calls whose record is whole, with the bound above for each."""
    fit = torch.from_numpy(np.random.default_rng(a + r).standard_normal(n).astype(np.float32)).cuda()
    g = hses_gpu.es_update(fit, 0, KEY, r, 0.02, 0, 0, a, b, 1.0)
    ref = torch.zeros((a, b), dtype=torch.float64, device="cuda")
    step = (n // 4 + 1) // 2 * 2  # whole pairs
    for lo in range(0, n, step):
        ref += hses_gpu.es_update(fit[lo:lo + step].contiguous(), lo, KEY, r, 0.02, 0, 0, a, b, 1.0).double()
    assert n * r * (a + b) * 2 > 512 << 20 > step * r * (a + b) * 2
    K = n * r // 2
    tol = 2 * (2.0 ** -20 + 2.0 ** -24 * math.sqrt(K)) * math.sqrt(K) * float((ref ** 2).mean().sqrt())
    assert float((g.double() - ref).abs().max()) <= tol
