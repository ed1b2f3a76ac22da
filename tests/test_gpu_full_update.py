"""Dense-leaf updates at the edges of the reduction's lanes and of the pairs' splits.

Bound: the f32 terms are summed in double, rounded to f32 and scaled in f32: two
roundings, 2^-23 of the result, and n 2^-53 of the sum of |terms|."""
import math

import numpy as np
import pytest
import torch

from hyperscalees_amd import _lib
from tests.test_gpu_dense import KEY, dense_grad_f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tid_lo,a,b,small", [
    (30, 0, 1, 1, False),      # 15 splits: one lane an element
    (31, 0, 3, 11, False),     # 16 splits, a partial block of elements
    (60, 1, 1, 33, False),     # 31 pairs: the second turn of a lane is ragged
    (200, 0, 64, 64, False),   # a split for each pair
    (200, 0, 64, 64, True),    # the workspace of 4096 threads
])
def test_full_update_lanes(hses_gpu, n, tid_lo, a, b, small):
    fit = np.random.default_rng(n + b).standard_normal(n).astype(np.float32)
    scale = np.float32(-math.sqrt(n) / n)
    f = torch.from_numpy(fit).cuda()
    if small:
        work = torch.empty(32 * a * b, dtype=torch.float64, device="cuda")
        g = torch.empty((a, b), device="cuda")
        _lib.call("hses_full_update", f.data_ptr(), n, tid_lo, KEY & (2 ** 64 - 1), 0.02, 0, 0, a, b,
                  float(scale), 0, g.data_ptr(), work.data_ptr(), work.numel() * 8,
                  torch.cuda.current_stream().cuda_stream)
    else:
        g = hses_gpu.full_update(f, tid_lo, KEY, 0.02, 0, 0, a, b, scale)
    ref = dense_grad_f64(fit, tid_lo, 0.02, KEY, a, b)
    mag = sum(np.abs(dense_grad_f64(fit[m:m + 1], tid_lo + m, 0.02, KEY, a, b)) for m in range(n))
    err = np.abs(g.cpu().numpy() - ref * float(scale))
    assert (err <= 2.0 ** -23 * np.abs(ref * scale) + n * 2.0 ** -53 * mag * abs(float(scale)) + 1e-30).all()
