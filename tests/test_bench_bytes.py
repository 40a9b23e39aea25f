"""The byte model of the benchmark's per-kernel rates: bytes that a launch moves,
so that launches without work are not credited with any."""
import os
import sys
from types import SimpleNamespace

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def grid(n1, n2, n3):
    return SimpleNamespace(cfg=SimpleNamespace(n1=n1, n2=n2, n3=n3, ng=4, recon=2))


@pytest.mark.parametrize("n,launches", [((256, 128, 64), 2), ((64, 64, 1), 1), ((7, 32, 16), 1)])
def test_ghosts_are_counted_once_for_the_launches_that_fill_them(n, launches):
    # launches: those a substep's boundary bytes are spread over (3-D, merged: the second ends at once;
    # the direction-by-direction pass does all of it in each of its two)
    g = grid(*n)
    ghosts = 1
    for x in n:
        ghosts *= x + 8 * (x > 1)
    ghosts -= n[0] * n[1] * n[2]
    assert bench.algorithmic_bytes(g, "bound") * launches == ghosts * 128


def test_averaging_without_failed_zones_moves_nothing():
    assert bench.algorithmic_bytes(grid(256, 128, 64), "fixup") == 0
    assert bench.algorithmic_bytes(grid(64, 64, 1), "fixup") == 0
    assert bench.algorithmic_bytes(grid(7, 32, 16), "fixup") == 7 * 32 * 16 * 4
