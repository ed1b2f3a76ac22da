"""Size queries of the library are kept per device: a device with more compute units needs
more workspace slots for the same shape."""
from hyperscalees_amd import _lib
from hyperscalees_amd import kernels as K


def test_size_of_each_device(monkeypatch):
    current, asked = [0], []

    def query(*shape):
        asked.append((current[0], shape))
        return 1000 * (current[0] + 1) + shape[0]

    monkeypatch.setattr(K, "_SIZES", {})
    monkeypatch.setattr(K, "_device", lambda: current[0], raising=False)
    monkeypatch.setattr(_lib, "fn", lambda name: query)
    got = []
    for current[0] in (0, 1, 0, 1):
        got.append(K._size("hses_perturbed_linear_workspace", 7, 8))
    assert got == [1007, 2007, 1007, 2007]
    assert asked == [(0, (7, 8)), (1, (7, 8))]
