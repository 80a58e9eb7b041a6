"""The fit kernel's splits: realizations 64 a workgroup, observations 8 a wave
and 240 a pass, wells 32 a tile.  Sizes on their edges, bit for bit against
the oracle, which fits one realization at a time."""
import numpy as np
import pytest

import oracle as O
from onekapy_amd import fit_and_draw
from onekapy_amd.model import RangeError

pytestmark = pytest.mark.gpu


def _site(nw, nobs, R, seed):
    rng = np.random.default_rng(seed)
    wxy = rng.uniform(0, 8000, (nw, 2))
    obs = [(float(x), float(y), float(z), 0.1)
           for x, y, z in zip(*rng.uniform(0, 8000, (2, nobs)), rng.uniform(8, 60, nobs))]
    d = dict(K=rng.lognormal(2.3, 0.5, R), b=rng.uniform(20, 30, R),
             q=rng.uniform(100, 1500, (R, nw)), z=rng.standard_normal((R, 6)))
    return wxy, obs, d


@pytest.mark.parametrize("nw,nobs,R", [(1, 6, 1), (32, 8, 63), (33, 9, 64), (31, 63, 65),
                                       (5, 65, 130), (2, 240, 3), (33, 241, 65)])
def test_fit_splits_bit_exact_vs_oracle(gpu_ctx, nw, nobs, R):
    wxy, obs, d = _site(nw, nobs, R, 1000 * nw + nobs)
    if R == 65:
        d["b"][3] = 1e4       # every head below the aquifer's top
        d["K"][5] = 1e-70     # standard deviations outside the short quotients' range
    ev, cov, coef = fit_and_draw(wxy, 4000.0, 4000.0, 0.0, obs, d["K"], d["b"], d["q"], d["z"])
    for r in sorted({0, 3, 5, 62, 63, 64, R - 1} & set(range(R))):
        om = O.OracleModel(0.0, d["K"][r], 0.25, d["b"][r],
                           np.c_[wxy, np.full(nw, 0.25), d["q"][r]])
        oev, ocov = om.fit(np.array(obs), 4000.0, 4000.0, O.MATH_CR)
        assert np.array_equal(np.ravel(oev), ev[r]), r
        assert np.array_equal(np.asarray(ocov).reshape(6, 6), cov[r]), r
        assert np.array_equal(O.mvn(oev, ocov, d["z"][r]), coef[r]), r


@pytest.mark.parametrize("bad", [0, 7, 8, 64, 240])
def test_fit_reports_an_observation_out_of_range_wherever_it_is(gpu_ctx, bad):
    wxy, obs, d = _site(3, 241, 65, 5)
    obs[bad] = obs[bad][:2] + (-1.0, 0.1)
    with pytest.raises(RangeError):
        fit_and_draw(wxy, 4000.0, 4000.0, 0.0, obs, d["K"], d["b"], d["q"], d["z"])
