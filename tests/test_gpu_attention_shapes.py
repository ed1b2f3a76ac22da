"""The spiking attention's stages at the edges of their instances, bit for bit against
the oracle: head sizes with registers of their own (8, 16, 32) at ragged token counts,
the general form at the largest head, and the encoder with rows of four columns, rows
that are not, and planes off 16 bytes."""
import numpy as np
import pytest
import torch

from hyperscalees_amd import _lib
from hyperscalees_amd import kernels as K
from tests import oracle_lib as O
from tests.test_gpu_attention import dev, test_attention_stage_bit_exact as check_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,H,hd", [
    (64, 4, 8), (9, 2, 8), (17, 3, 16), (1, 1, 16), (64, 2, 32), (33, 1, 32), (64, 1, 64), (16, 2, 1),
])
def test_attention_head_sizes(hses_gpu, R, H, hd):
    check_attention(hses_gpu, R, H, hd)


@pytest.mark.parametrize("R,d,T,shared,shift", [
    (5, 12, 7, False, 0),    # four columns a thread, steps not a multiple of four
    (5, 12, 3, True, 0),     # one embedding for all members
    (3, 10, 5, False, 0),    # one column a thread
    (5, 12, 4, True, 1),     # planes 4 bytes past a 16-byte boundary
])
def test_encode_forms(hses_gpu, R, d, T, shared, shift):
    rng = np.random.default_rng(R * d + T)
    n = 70                   # members past a block's rows
    M = n * R

    def shifted(a):
        t = torch.empty(a.size + shift, dtype=torch.float32, device="cuda")
        t[shift:].copy_(dev(a).reshape(-1))
        return t[shift:]

    cur = [rng.normal(0.4, 0.4, (T, M, d)).astype(np.float32) for _ in range(3)]
    th = [rng.uniform(0.03, 0.08, n).astype(np.float32) for _ in range(3)]
    pos = rng.standard_normal((1 if shared else n, R, d)).astype(np.float32)
    cd, thd, posd = [shifted(c) for c in cur], [dev(t) for t in th], shifted(pos)
    X = shifted(np.zeros((M, d), np.float32))
    _lib.call("hses_sa_encode", K._p(cd[0]), K._p(cd[1]), K._p(cd[2]), T, M, d, R, K._p(thd[0]),
              K._p(thd[1]), K._p(thd[2]), 20.0, K._p(posd), int(not shared), K._p(X), K._stream())
    got = X.cpu().numpy().reshape(M, d)
    for m in range(n):
        rows = slice(m * R, (m + 1) * R)
        ref = np.zeros((R, d), np.float32)
        O.load().or_sa_encode(*[np.ascontiguousarray(c[:, rows]) for c in cur], T, R, d,
                              *[float(t[m]) for t in th], 20.0,
                              np.ascontiguousarray(pos[0 if shared else m]), ref)
        np.testing.assert_array_equal(got[rows], ref, err_msg=f"member {m}")
