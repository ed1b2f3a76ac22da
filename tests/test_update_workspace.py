"""The ES update's workspace of layers whose record of normals runs in parts: the partial
sums of one part at a time and the record's bound, not a partial for every part."""
import pytest

from hyperscalees_amd import _lib


@pytest.mark.parametrize("n,rank", [(1 << 16, 16), (1 << 20, 31)])
def test_workspace_of_a_large_layer(n, rank):
    a = b = 8192
    size = _lib.load().hses_es_update_workspace(a, b, rank, n)
    # the record: whole K chunks of 32 and two pairs past its 512 MB
    assert size <= (520 << 20) + 4 * a * b + 16, f"{size / 2 ** 30:.1f} GiB"
