"""The FP64-exact rasterizer's outer chords: whatever rule a segment, an umbra
or a lattice falls under, the marked nodes are the oracle's."""
import numpy as np
import pytest

import oracle as O
from onekapy_amd import _lib

pytestmark = pytest.mark.gpu

# spacing, umbra, origin, longest step in umbras: the usual case; windows of
# more than 32 and 64 columns; spacing above the umbra; above 1,000 umbras (no
# chords); coordinates whose rounding reaches the chords' slack (no chords);
# steps above 1,000 umbras (no chords); nodes on the umbra circle itself
RULES = {
    "two_cells": (20.0, 40.0, 1234.5, 0.25),
    "wide_umbra": (5.0, 300.0, -77.25, 0.5),
    "coarse": (40.0, 15.0, 3.0, 2.0),
    "spacing_above_1000_umbras": (2000.0, 1.5, 10.0, 300.0),
    "huge_coordinates": (4096.0, 8192.0, 1.0e15, 0.5),
    "step_above_1000_umbras": (5.0, 0.75, 50.0, 2000.0),
    "lattice_points": (8.0, 24.0, 0.0, None),
}


@pytest.mark.parametrize("case", sorted(RULES))
def test_outer_chords_mark_the_oracles_nodes(gpu_ctx, case):
    spacing, umbra, origin, step = RULES[case]
    rng = np.random.default_rng(sorted(RULES).index(case))
    n = 150
    half = 0.5 * n * spacing
    field = O.OracleField(spacing, spacing, origin, origin)
    field.expand(origin - half, origin + half, origin - half, origin + half)
    pts = [np.array([origin, origin])]
    for k in range(300):
        p = pts[-1].copy()
        kind = k % 8
        if step is None:                       # from lattice point to lattice point
            p += spacing * rng.integers(-3, 4, 2)
        elif kind == 0:                        # along an axis
            p[rng.integers(0, 2)] += rng.uniform(-1, 1) * step * umbra
        elif kind == 1:                        # no length, or hardly any
            p += rng.uniform(-1, 1, 2) * umbra * (0.0 if k % 16 else 1e-9)
        elif kind == 2:                        # nearly along an axis
            p += np.array([1.0, 1e-7 * rng.uniform(-1, 1)])[rng.permutation(2)] * step * umbra
        else:
            a = rng.uniform(0, 2 * np.pi)
            p += rng.uniform(0, 1) * step * umbra * np.array([np.cos(a), np.sin(a)])
        pts.append(np.clip(p, origin - 0.98 * half, origin + 0.98 * half))
    xy = np.ascontiguousarray(pts)
    s = field.s
    grid = _lib.make_grid(s.xmin, s.ymin, s.xmax, s.ymax, spacing, spacing, s.nrows, s.ncols)
    marks = np.zeros(field.shape, dtype=np.uint8)
    gpu_ctx.check(gpu_ctx.lib.oka_rasterize(gpu_ctx.h, grid, xy.shape[0], _lib.ptr(xy),
                                            float(umbra), _lib.ptr(marks), 0))
    before = field.shape
    field.rasterize(xy, umbra)
    assert field.shape == before
    assert field.rgrid.any()
    assert np.array_equal(marks.astype(bool), field.rgrid)
