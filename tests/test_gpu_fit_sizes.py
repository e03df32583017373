"""The Gaussian fit and bisector at the sizes where its wave can go wrong: velocity
counts around the 64 lanes, around the three points a lane keeps in flight (192) and at
the largest, with unit and per-point errors, against the oracle's fit of the same CCFs.
Both stop at xtol = 1e-8, so they agree to that in the parameters: 1e-7 relative in
continuum and contrast, 1e-4 m/s in RV, FWHM and span (the bars of the parity tests)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_v", [41, 63, 64, 65, 128, 129, 191, 192, 193, 385, 1023, 1024])
@pytest.mark.parametrize("errors", [False, True])
def test_fit_sizes(engine, n_v, errors):
    rng = np.random.default_rng(n_v)
    v = np.linspace(-20000.0, 20000.0, n_v)
    v0, fw, k = rng.uniform(-1500, 1500, 5), rng.uniform(7e3, 11e3, 5), rng.uniform(0.3, 0.6, 5)
    u = (v - v0[:, None]) / (fw[:, None] / 2.3548200450309493)
    y = 1.0 - k[:, None] * np.exp(-0.5 * u * u) * (1.0 + 0.01 * u)
    err = np.exp(rng.uniform(-0.3, 0.3, y.shape)) if errors else None
    got = engine.fit_ccf_host(v, y, err)
    for i in range(5):
        ref = O.fit_ccf(v, y[i]) if err is None else O.fit_ccf(v, y[i], err[i])
        par = got["par"][i]
        assert np.all(np.abs(par[:2] - ref["par"][:2]) <= 1e-7 * np.abs(ref["par"][:2]))
        assert np.all(np.abs(par[2:] - ref["par"][2:]) <= 1e-4), (par, ref["par"])
        assert np.max(np.abs(got["model"][i] - ref["model"])) <= 1e-7
