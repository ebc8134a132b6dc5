"""How much page-locked memory a context keeps for a host state."""
import pytest

from sph_amd import _native as N


@pytest.mark.parametrize("n,want", [(0, 4096), (1, 4096), (73, 4352), (2999, 168448), (74000, 256 + 56 * 74000 + 128),
                                    (100000, 4 << 20), (300000, 4 << 20), (700000, 4900032 // 512 * 512), (4200000, 16 << 20)])
def test_pinned_bytes(n, want):
    nbytes = 256 + 56 * n
    got = N.pinned_bytes(nbytes)
    assert got == want and got % 256 == 0
    assert got <= max(4 << 20, nbytes // 8)  # a new context of 300,000 particles locked 16 MiB


def test_the_bound_holds(monkeypatch):
    monkeypatch.setattr(N, "PINNED_BYTES", 8448)
    assert [N.pinned_bytes(256 + 56 * n) for n in (1, 100, 2999, 10 ** 7)] == [4096, 5888, 8448, 8448]
