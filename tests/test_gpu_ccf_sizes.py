"""The mask CCF in calls of few, some and many phases (three forms of the kernel: rounds of
lines with lanes sharing a velocity, loads ahead, plain; 33 chunks of lines give 297 spectrum
chunks, 264 and 528 blocks): a phase's CCF has the same bits in each, and the smallest call's
equals the oracle's CCF of its spectra (the bar of the parity tests, 1e-12).  At velocity
counts on both sides of 4, 2 and 1 lanes per velocity, and with line footprints from 100
pixels to past the 512 and 2048 of the staged rows, lines at both ends of the spectrum and a
last chunk of one line."""
import numpy as np
import pytest

from soap_gpu_amd import synth
from soap_gpu_amd.engine import Engine, setup_workload
from tests.pipeline_ref import ccf_stage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_v,half", [(81, 20e3), (254, 20e3), (257, 20e3), (401, 100e3), (510, 64e3), (513, 20e3),
                                      (161, 80e3), (161, 400e3), (1022, 400e3), (33, 15e3)])
def test_ccf_bits_do_not_depend_on_the_call(n_v, half):
    n, n_lines = 9000, 1025
    rng = np.random.default_rng(n_v)
    w = synth.small(seed=5, grid=24, n=n, n_mu=3, n_phase=45, n_lines=40, lmin=5000.0,
                    lmax=5000.0 * np.exp((n - 1) * 1e-6))
    w.vgrid = np.linspace(-half, half, n_v)
    w.mask_l = rng.uniform(w.wave[211], w.wave[-212], n_lines)  # in no order, windows over both ends
    w.mask_w = rng.uniform(0.11, 0.9, n_lines)
    phases, regions = w.phases, w.regions
    got = {}
    for p in (2, 20, 45):
        w.phases, w.regions = phases[:p], regions[:p]
        e = Engine(0)
        setup_workload(e, w)
        e.run_series(w.star, w.sigma_inst)
        frames = [0, 1, -1]
        lower = np.stack([[e.get_lower(f, t) for t in range(3)] for f in frames])
        got[p] = lower, e.get_ccf()[frames]
        if p == 2:
            ref = ccf_stage(w, lower)["ccf"]
            np.testing.assert_allclose(got[p][1], ref, rtol=1e-12, atol=1e-13)
        e.close()
    for p in (20, 45):
        np.testing.assert_array_equal(got[p][0], got[2][0])
        np.testing.assert_array_equal(got[p][1], got[2][1])
