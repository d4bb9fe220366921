"""bench.py's account of the kernels a plan runs (CPU)."""
import os
import sys
from types import SimpleNamespace

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


class _Plan:
    """A plan of which the first n slices are matrix-core items (32 x 32 tiles)."""

    def __init__(self, n):
        self.n = n

    def info(self, s):
        return {"tile_w": 32 if s < self.n else 64}


@pytest.mark.parametrize("n,slices,spec_tile,tile,share", [
    (64, 64, 0, -1, 1.0), (64, 80, 0, -1, 0.8), (64, 64, -1, 0, 1.0),
    (0, 64, 0, -1, 0.0),                       # a stack too small for the matrix cores
    (64, 64, 2, -1, 0.0), (64, 64, -1, 2, 0.0)])   # 32 x 32 tiles that were asked for
def test_roofline_follows_the_plan(n, slices, spec_tile, tile, share):
    args = SimpleNamespace(interp="linear", store="f32", lds_half=0, slices_per_item=0, tile=tile)
    specs = [SimpleNamespace(tile=spec_tile)] * slices
    got = bench.matrix_core_share(_Plan(n), specs, [(512, 450)] * slices, args)
    assert got == pytest.approx(share)
    roof = bench.roofline_of(args, slices, 60.0, None, got)
    assert roof["bound"] == ("mfma" if share else "valu")
    if share:
        assert roof["mfma_executed"] == pytest.approx(60.0 * share * 64 / bench.FLOP_PER_UPDATE)
