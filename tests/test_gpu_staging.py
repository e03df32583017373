"""Results through the shared pinned staging: many contexts on many threads at once, more
than the staging has buffers, and results larger than a buffer, each equal to the same
call made alone; and a single output equal to its part of the whole."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from soap_gpu_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _call(n_ccf, seed, n_v=161):
    rng = np.random.default_rng(seed)
    v = np.linspace(-20000.0, 20000.0, n_v)
    u = (v - rng.uniform(-1500, 1500, (n_ccf, 1))) / 3500.0
    y = 1.0 - rng.uniform(0.3, 0.6, (n_ccf, 1)) * np.exp(-0.5 * u * u) * (1.0 + 0.01 * u)
    eng = Engine(0)
    try:
        return [eng.fit_ccf_host(v, y) for _ in range(3)]
    finally:
        eng.close()


# 3000 CCFs of 161 velocities need 10 MB of results: past the largest buffer
@pytest.mark.parametrize("sizes", [[1, 3, 40, 99] * 4, [3000, 7]])
def test_many_contexts_share_the_staging(sizes):
    import torch  # noqa: F401
    alone = [_call(n, i)[0] for i, n in enumerate(sizes)]
    with ThreadPoolExecutor(max_workers=12) as ex:
        for ref, got in zip(alone, ex.map(lambda a: _call(a[1], a[0]), list(enumerate(sizes)))):
            for g in got:
                assert all(np.array_equal(g[k], ref[k]) for k in ref)


def test_one_output_of_the_fit(engine):
    from soap_gpu_amd import synth
    from soap_gpu_amd.engine import setup_workload
    w = synth.small(n_phase=3)
    setup_workload(engine, w)
    engine.run_series(w.star, w.sigma_inst)
    whole = engine.get_fit()
    dp = ctypes.POINTER(ctypes.c_double)
    for i, k in enumerate(("par", "model", "depth", "bis")):
        out = np.zeros(whole[k].size)
        args = [None] * 4
        args[i] = out.ctypes.data_as(dp)
        assert engine.L.soap_get_fit(engine.ctx, *args) == 0
        assert np.array_equal(out.reshape(whole[k].shape), whole[k])


def test_refused_forward_gives_its_staging_back():
    """A forward of the differentiable model that is refused after its targets are on their
    way (a resolution window too wide for the LDS), then calls that use the same staging."""
    import torch
    from soap_gpu_amd import synth
    from soap_gpu_amd.diff import DiffModel
    from soap_gpu_amd.engine import SoapError, select_mask_lines
    ref = _call(7, 0)[0]
    n, p = 24000, 3
    w = synth.small(seed=4, grid=24, n=n, n_mu=4, n_phase=1, n_lines=30, lmin=5000.0, lmax=5000.0 * np.exp((n - 1) * 1e-6))
    sl, sw = select_mask_lines(w.wave, w.mask_l, w.mask_w, 210)
    dev = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")  # noqa: E731
    q, maps, target = dev(w.cubes["q"]), dev(np.full((p, 8, 8), 0.2)), dev(np.full((p, n), 400.0))
    eng = Engine(0)
    wide, narrow = (DiffModel(eng, w.wave, w.mu_bounds, sl, sw, w.vgrid, 24, p, 8, s, 210) for s in (65000.0, w.sigma_inst))
    args = ([2.0, 0.29, 0.34, 0.3], q, q, maps, target, np.arange(3.0), np.full(p, 9e3), 1e-6, 1e-3, 1e-5)
    loss = narrow.forward(*args)[0]
    for _ in range(3):
        eng._chk(eng.L.soap_diff_setup(eng.ctx, 24, p, 8, 65000.0, None), "diff_setup")
        with pytest.raises(SoapError, match="too wide"):
            wide.forward(*args)
        got = _call(7, 0)[0]
        assert all(np.array_equal(got[k], ref[k]) for k in ref)
        eng._chk(eng.L.soap_diff_setup(eng.ctx, 24, p, 8, float(w.sigma_inst), None), "diff_setup")
        assert narrow.forward(*args)[0] == loss
    eng.close()
