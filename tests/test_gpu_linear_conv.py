"""The linear grids' resolution convolution where a pixel stands out: its sums end where the
rest of the window is below their rounding, which values that are not finite, or far
larger than the others, must not be.  The convolved spectra against the oracle's of the
same raw spectra: the same pixels not finite, the others to 1e-11 of themselves (the
sums' terms have one sign there; a width's rounding moves a Gaussian factor at 30 widths
by 450 of its relative 2e-16, with the oracle's and the recurrence's own about 1e-12)."""
import numpy as np
import pytest

import oracle as O
from soap_gpu_amd import synth
from soap_gpu_amd.engine import Engine, setup_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 1e12, 1e30, 1e200])
@pytest.mark.parametrize("at", [700, 1535])
def test_pixel_that_stands_out(value, at):
    w = synth.linear_small(seed=3, grid=24, n=2611, n_mu=3, n_phase=1)
    e = Engine(0)
    setup_workload(e, w, with_mask=False)
    e.quiet_star()
    q, qs = e.get_quiet(0), e.get_quiet(1)
    raw = np.zeros(w.n)
    raw[at] = value
    e.alloc_phases(1)
    e.set_raw(0, raw, raw, raw)
    e.resolution(w.sigma_inst)
    for t in range(3):
        got = e.get_lower(0, t)
        ref, _ = O.lower_resolution(O.GRID_LINEAR, w.wave, w.sigma_inst, q if t == 1 else qs, raw, 1)
        np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
        ok = np.isfinite(ref) & (ref != 1.0)
        assert np.max(np.abs(got[ok] - ref[ok]) / np.abs(ref[ok]), initial=0.0) <= 1e-11  # +inf: nothing is finite
    e.close()
