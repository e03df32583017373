"""The linear gathers' two interpolation forms against the oracle's per-cell sums (the
spectra's bar, 1e-12 norm-wise on the interior): a grid of the step itself (quiet star through
taps, active cells by runs; at large wavelengths and by groups the reciprocal form), one whose
differences stray from the step by 5e-9 (the reciprocal form by columns) and one that strays by
1e-4 (the division), under solid-body rotation (by columns) and differential rotation (by
groups); pixel counts off the 256-pixel tiles."""
import numpy as np
import pytest

from soap_gpu_amd import synth
from soap_gpu_amd.engine import GRID_LINEAR, setup_workload
from tests.pipeline_ref import normwise, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmin,stray,w_ratio,n", [(5000.0, 0.0, 0.0, 3001), (15000.0, 0.0, -0.2, 2817),
                                                   (5000.0, 5e-9, 0.0, 2600), (5000.0, 1e-4, 0.0, 2900),
                                                   (5000.0, 1e-4, -0.2, 2563)])
def test_linear_forms(engine, lmin, stray, w_ratio, n):
    w = synth.linear_small(seed=21, grid=40, n=n, n_mu=5, n_phase=2, lmin=lmin)
    assert w.grid_kind == GRID_LINEAR
    w.star["w_ratio"] = w_ratio
    if stray:
        rng = np.random.default_rng(2)
        w.wave[1:] += 0.005 * stray * rng.uniform(-0.5, 0.5, n - 1)
    o = run_oracle(w, with_ccf=False)
    setup_workload(engine, w, with_mask=False)
    engine.quiet_star()
    engine.integrate()
    for i in range(2):
        assert normwise(engine.get_quiet(i), o["quiet"][i]) <= 1e-12
    for p in range(2):
        for got, ref in zip(engine.get_raw(p), o["raw"][p]):
            assert normwise(got, ref) <= 1e-12


@pytest.mark.parametrize("speed,n", [(0.1, 2561), (2.0, 2815), (6.0, 3001), (9.0, 3001), (14.0, 3001)])
def test_linear_quiet_reach(engine, speed, n):
    """The quiet star by columns from windows of a few pixels to ones too wide for the taps (the
    rotation sped up), against the oracle.  Bar: both sides' weights may be off by one unit in the
    last place of a shifted wavelength, so by ulp(lambda) / step of the row's change per pixel."""
    w = synth.linear_small(seed=21, grid=40, n=n, n_mu=5, n_phase=2)
    w.star["prot"] /= speed
    o = run_oracle(w, with_ccf=False)
    setup_workload(engine, w, with_mask=False)
    engine.quiet_star()
    limb = np.abs(o["maps"]["limb"][o["maps"]["limb"] != -999.0]).sum()
    for i, k in enumerate(("q", "qsed")):
        change = np.abs(np.diff(w.cubes[k], axis=1)).max() * limb / np.abs(o["quiet"][i]).max()
        assert normwise(engine.get_quiet(i), o["quiet"][i]) <= 2 * np.spacing(w.wave[-1]) / 0.005 * change
