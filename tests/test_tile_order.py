"""The large-M kernels' tile order (tile_coords of csrc/gemm_main.h), restated: every tile once, whatever
the counts, and contiguous ranges per XCD where they are kept."""
import pytest

GROUP_M = 8


def _coords(t, nbm, nbn, start):
    n = nbm * nbn
    if start == 0 or n % 8 == 0 or nbm <= GROUP_M or nbn >= start:
        t = (t & 7) * (n >> 3) + min(t & 7, n & 7) + (t >> 3)
    g, r = divmod(t, GROUP_M * nbn)
    rows = min(nbm - g * GROUP_M, GROUP_M)
    return g * GROUP_M + r % rows, r // rows


@pytest.mark.parametrize("start", [0, 14, 28])
def test_every_tile_once(start):
    for nbm in (1, 2, 7, 8, 9, 16, 25, 33):
        for nbn in (1, 5, 8, 13, 14, 27, 28, 31):
            seen = {_coords(t, nbm, nbn, start) for t in range(nbm * nbn)}
            assert seen == {(m, n) for m in range(nbm) for n in range(nbn)}, (nbm, nbn)
