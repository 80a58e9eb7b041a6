"""The workgroup schedule's launch shapes: whatever lanes a realization's
particles are given, the counts, per-trace statuses and statistics are those of
the pool, which deals out particles on its own."""
import numpy as np
import pytest

from onekapy_amd import Realizations, _lib, chronicle_into_field, start_points
from onekapy_amd.sites import fixed_field
from helpers import oracle_chronicle, oracle_fit_draw, small_site
from test_gpu_pool import STAT_KEYS, _both

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
# the fine lattices' bitmaps are tiled, (2, 1500) shared and (600, 20) a
# workgroup a realization
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


def _workgroup(s, d, coef, pf, precision, confined=True, **kw):
    real = Realizations(d["K"], d["n"], d["b"], d["q"], coef)
    return chronicle_into_field(pf, s.wells_xy(), s.xt, s.yt, real,
                                start_points(s.xt, s.yt, s.rt, s.npaths), s.duration, s.tol,
                                s.maxstep, s.umbra, precision=precision, confined=confined,
                                schedule=_lib.SCHED_WORKGROUP, **kw)


def _same(a, b):
    assert np.array_equal(a.counts, b.counts)
    assert np.array_equal(a.trace_status, b.trace_status)
    for k in STAT_KEYS:
        assert getattr(a.stats, k) == getattr(b.stats, k), k
    assert list(a.stats.status_count) == list(b.stats.status_count)


# more realizations than the GPU runs workgroups at once (at most 8 a CU), none
# shared (20 particles): the queue alone; tiled, a few slots that overflow, HBM
@pytest.mark.parametrize("mode,slots", [(_lib.BITMAP_TILED, 0), (_lib.BITMAP_TILED, 3),
                                        (_lib.BITMAP_HBM_FLAT, 0)])
@pytest.mark.parametrize("precision", [_lib.FP64_EXACT, _lib.FP32], ids=["fp64", "fp32"])
def test_queue_without_sharing(gpu_ctx, mode, slots, precision):
    s, d = small_site(nreal=3000, npaths=20)
    assert s.nrealizations > 8 * gpu_ctx.device_info()["num_cu"]
    _, _, coef = oracle_fit_draw(s, d)
    pf = fixed_field(s.xt, s.yt, 5.0, 900, 950)
    print(f"mode {mode} slots {slots} precision {precision}", flush=True)
    wg = _workgroup(s, d, coef, pf, precision, bitmap_mode=mode, tile_slots=slots)
    _, auto = _both(s, d, coef, pf, s.umbra, precision)
    _same(wg, auto)


# shared realizations whose bitmaps are flat in HBM, and tiled with overflow
@pytest.mark.parametrize("nreal,npaths", [(4, 600), (1500, 300)])
@pytest.mark.parametrize("mode,slots", [(_lib.BITMAP_HBM_FLAT, 0), (_lib.BITMAP_TILED, 2)])
@pytest.mark.parametrize("precision", [_lib.FP64_EXACT, _lib.FP32], ids=["fp64", "fp32"])
def test_shared_bitmaps_in_hbm(gpu_ctx, nreal, npaths, mode, slots, precision):
    s, d = small_site(nreal=nreal, npaths=npaths)
    _, _, coef = oracle_fit_draw(s, d)
    pf = s.fixed_field()
    print(f"{nreal} x {npaths} mode {mode} precision {precision}", flush=True)
    wg = _workgroup(s, d, coef, pf, precision, bitmap_mode=mode, tile_slots=slots)
    _, auto = _both(s, d, coef, pf, s.umbra, precision)
    _same(wg, auto)


# the unconfined field, whose traces may end at their start points (F lowered by
# 0.7 K b^2 / 2): they count among a shared realization's traces
@pytest.mark.parametrize("shift", [0.0, 0.7])
@pytest.mark.parametrize("precision", [_lib.FP64_EXACT, _lib.FP32], ids=["fp64", "fp32"])
def test_shared_unconfined_realizations(gpu_ctx, shift, precision):
    s, d = small_site(nreal=12, npaths=300, seed=11)
    _, _, coef = oracle_fit_draw(s, d)
    coef[:, 5] -= shift * 0.5 * d["K"] * d["b"] ** 2
    pf = s.fixed_field()
    print(f"shift {shift} precision {precision}", flush=True)
    _, wg = _both(s, d, coef, pf, s.umbra, precision, confined=False)
    if shift > 0:
        assert 0 < wg.stats.status_count[_lib.TRACE_TRUNCATED] < s.nrealizations * s.npaths
    if precision == _lib.FP64_EXACT:
        ocounts, ost = oracle_chronicle(s, d, coef, pf, confined=False)
        assert np.array_equal(wg.counts, ocounts)
        assert list(wg.stats.status_count) == list(ost[2:6])


# 1,300 merged bitmaps of 4,600^2 nodes and as many overflow regions are over
# the limit on them: nothing is shared
@pytest.mark.parametrize("precision", [_lib.FP64_EXACT, _lib.FP32], ids=["fp64", "fp32"])
def test_too_large_to_share(gpu_ctx, precision):
    s, d = small_site(nreal=1300, npaths=257)
    s.duration /= 10.0
    _, _, coef = oracle_fit_draw(s, d)
    pf = fixed_field(s.xt, s.yt, 5.0, 4600, 4600)
    print(f"precision {precision}", flush=True)
    _both(s, d, coef, pf, s.umbra, precision)
