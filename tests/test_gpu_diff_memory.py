"""Device memory of a differentiable model of the full disk (grid 1000, 20 bins, faculae)
over forward and backward: no more than its four phase spectra, 40 bytes per cell of the
disk and a correlation partial per 2304 pixels, which is what the per-cell form held, and
8 % for allocation."""
import numpy as np
import pytest

from soap_gpu_amd import synth

pytestmark = pytest.mark.gpu


def test_memory_of_a_full_disk():
    import torch
    from soap_gpu_amd.diff import DiffModel
    from soap_gpu_amd.engine import Engine, select_mask_lines
    n, grid, P, n_mu, M, vsini, h = 100000, 1000, 64, 20, 32, 3.0, 1e-6
    w = synth.small(seed=4, grid=grid, n=n, n_mu=n_mu, n_phase=1, n_lines=30, lmin=5000.0,
                    lmax=5000.0 * np.exp((n - 1) * h))
    sl, sw = select_mask_lines(w.wave, w.mask_l, w.mask_w, 210)
    dev = torch.device("cuda")
    q, s, f = (torch.tensor(w.cubes[k], dtype=torch.float64, device=dev) for k in ("q", "sp", "fac"))
    maps = torch.full((P, M, M), 0.2, dtype=torch.float64, device=dev)
    target = torch.full((P, n), 5e5, dtype=torch.float64, device=dev)

    def used(grid, P):
        """Device bytes that the model takes, after a forward and a backward."""
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        before = torch.cuda.mem_get_info()[0]
        eng = Engine(0)
        model = DiffModel(eng, w.wave, w.mu_bounds, sl, sw, w.vgrid, grid, P, M, w.sigma_inst, 210, lb=w.star["lb"])
        model.forward([vsini, 0.29, 0.34, 0.3, 1.1], q, s, maps[:P], target[:P], np.zeros(P), np.zeros(P), 1e-9, 0.0, 0.0,
                      f=f, fmaps=maps[:P])
        grads = model.backward()
        del grads
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        after = torch.cuda.mem_get_info()[0]
        eng.close()
        return before - after

    used(24, 2)  # what the runtime takes once
    got = used(grid, P)
    nd = 2 * int(np.ceil(vsini * 1e3 / 299792458.0 / h)) + 5
    held = 8 * (4 * P * n + 5 * grid * grid + P * n_mu * 3 * nd * -(-n // 2304))
    assert got <= 1.08 * held, (got / 1e6, held / 1e6)
