"""The workgroup schedule's launch shapes: whatever lanes a realization's
particles are given, the counts, per-trace statuses and statistics are those of
the pool, which deals out particles on its own."""
import pytest

from onekapy_amd import _lib
from onekapy_amd.sites import fixed_field
from helpers import oracle_fit_draw, small_site
from test_gpu_pool import _both

pytestmark = pytest.mark.gpu


# a lone particle; a wave and one more; whole waves; the largest workgroup and
# the first refilled lane
@pytest.mark.parametrize("npaths", [1, 64, 65, 192, 256, 257])
@pytest.mark.parametrize("precision", [_lib.FP64_EXACT, _lib.FP32], ids=["fp64", "fp32"])
def test_lanes_for_the_particles(gpu_ctx, npaths, precision):
    s, d = small_site(nreal=6, npaths=npaths)
    _, _, coef = oracle_fit_draw(s, d)
    print(f"npaths {npaths} precision {precision}", flush=True)
    _both(s, d, coef, s.fixed_field(), s.umbra, precision)


# (realizations, particles, field spacing): one realization spread over many
# workgroups; fewer realizations than CUs; every workgroup's last one shared;
# the fine lattices' bitmaps are tiled
@pytest.mark.parametrize("nreal,npaths,spacing", [
    (1, 257, None), (1, 3000, None), (3, 1000, None), (700, 320, None), (2500, 300, None),
    (2, 1500, 5.0), (600, 20, 5.0)])
@pytest.mark.parametrize("precision", [_lib.FP64_EXACT, _lib.FP32], ids=["fp64", "fp32"])
def test_shared_realizations(gpu_ctx, nreal, npaths, spacing, precision):
    s, d = small_site(nreal=nreal, npaths=npaths)
    _, _, coef = oracle_fit_draw(s, d)
    pf = s.fixed_field() if spacing is None else fixed_field(s.xt, s.yt, spacing, 900, 950)
    print(f"{nreal} x {npaths} spacing {spacing} precision {precision}", flush=True)
    _both(s, d, coef, pf, s.umbra, precision)


# lattices (nodes a side) whose tile index leaves 8, 4 and 3 workgroups' LDS
# enough slots, that of 2 only, and hardly any
@pytest.mark.parametrize("nside,npaths", [(700, 40), (1500, 40), (1500, 300), (2900, 200),
                                          (3300, 70), (3550, 30)])
def test_tiles_for_the_workgroups(gpu_ctx, nside, npaths):
    s, d = small_site(nreal=5, npaths=npaths)
    _, _, coef = oracle_fit_draw(s, d)
    pf = fixed_field(s.xt, s.yt, 6000.0 / nside, nside, nside)
    print(f"nside {nside} npaths {npaths}", flush=True)
    _both(s, d, coef, pf, s.umbra, _lib.FP64_EXACT)
