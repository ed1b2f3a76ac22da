"""The LIF scan to bits over runs of rows, bit for bit: widths around the words' edges,
rows that leave one to three columns at the plane's end, partial last blocks, scans of
several batches, a plane off 16 bytes, spike rows with a gap, and in-place potentials."""
import numpy as np
import pytest
import torch

from hyperscalees_amd import _lib
from hyperscalees_amd import kernels as K
from tests import oracle_lib as O
from tests.test_gpu_spiking import unpack_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,M,h,shift,gap", [
    (20, 37, 130, 0, 0),     # one column past two words, two columns left at the end
    (16, 101, 63, 1, 1),     # unaligned planes, three columns left
    (17, 45, 65, 2, 0),      # one column left
    (64, 9, 500, 0, 2),      # the longest scan, wide rows
    (3, 5, 511, 3, 0),       # widest with four rows a block; a block of one row
    (5, 700, 10, 0, 0),      # six rows a word
    (2, 4, 1, 1, 0),         # four columns in all
    (6, 225, 1, 0, 0),       # last blocks of one, two and three columns: most threads idle
    (5, 226, 1, 1, 0),
    (3, 77, 3, 0, 1),
    (7, 113, 2, 2, 0),
    (65, 6, 100, 0, 0),      # past the longest: the one-column kernel
    (4, 5, 513, 0, 0),       # too wide for a run: the one-column kernel
])
def test_lif_runs(hses_gpu, T, M, h, shift, gap):
    rng = np.random.default_rng(T + M + h)
    cur = (rng.standard_normal((T, M, h)) * 1.5 + 0.4).astype(np.float32)
    v0 = (rng.standard_normal((M, h)) * 0.3).astype(np.float32)
    ref_s, ref_v = O.lif(cur, 10.0, 0.8, v0)
    words = (h + 63) // 64 + gap
    ct = torch.zeros(cur.size + shift, device="cuda")
    vt = torch.zeros(v0.size + shift, device="cuda")
    ct[shift:].copy_(torch.from_numpy(cur).reshape(-1))
    vt[shift:].copy_(torch.from_numpy(v0).reshape(-1))
    out = torch.full((T, M, words), -1, dtype=torch.int64, device="cuda")
    _lib.call("hses_lif_scan", ct.data_ptr() + 4 * shift, vt.data_ptr() + 4 * shift, T, M, h, h, 10.0, 0.8,
              out.data_ptr(), K.FMT_BITS, words, vt.data_ptr() + 4 * shift, K._stream())
    np.testing.assert_array_equal(unpack_bits(out, words * 64)[..., :h], ref_s)
    tail = unpack_bits(out, words * 64)[..., h:(h + 63) // 64 * 64]
    assert not tail.any()                                   # bits past the row are 0
    assert (out.cpu().numpy()[..., words - gap:] == -1).all()   # the gap is not written
    got = vt.cpu().numpy()
    np.testing.assert_array_equal(got[shift:].view(np.uint32), ref_v.reshape(-1).view(np.uint32))
    assert not got[:shift].any()
