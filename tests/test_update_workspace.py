"""The ES update's workspace: where its record of normals runs in parts, the partial sums of
one part at a time and the record's bound; where the record is given, the partial sums alone."""
import pytest
import torch

from hyperscalees_amd import _lib
from hyperscalees_amd import kernels as K


@pytest.mark.parametrize("n,rank", [(1 << 16, 16), (1 << 20, 31)])
def test_workspace_of_a_large_layer(n, rank):
    a = b = 8192
    size = _lib.load().hses_es_update_workspace(a, b, rank, n)
    # the record: whole K chunks of 32 and two pairs past its 512 MB
    assert size <= (520 << 20) + 4 * a * b + 16, f"{size / 2 ** 30:.1f} GiB"


def test_workspace_of_an_update_from_a_record(monkeypatch):
    """The SNN-MLP's first layer (784 -> 128, rank 128, 8192 members): 512 splits at most."""
    asked = []
    monkeypatch.setattr(K, "_dev", lambda t, dtype, name: t)
    monkeypatch.setattr(K, "_stream", lambda: 0)
    monkeypatch.setattr(K, "_device", lambda: 0)
    monkeypatch.setattr(K, "_workspace", lambda nbytes, device: asked.append(nbytes) or torch.empty(0))
    monkeypatch.setattr(_lib, "call", lambda *args: 0)
    K.es_update_rec(torch.zeros(8192), 0, torch.zeros(1), 128, 0.02, 128, 784, 1.0)
    assert asked[0] <= 512 * 128 * 784 * 4 + 16
    assert _lib.load().hses_es_update_rec_workspace(128, 784, 16, 64) == 0  # refused below rank 32
