"""The differentiable model's kernels at the shapes where their tiles and lanes end:
phase counts around the 64 lanes and the group sizes, maps finer and coarser than the
disk grid and of sizes off the 16-node tiles, one and many bins, shifts of less than a
pixel and of many, with and without faculae.  The CCF terms are off, so the loss is the
spectra's, quadratic in the seed rows, the maps, the contrasts and the limb coefficients:
against the oracle's loss (1e-12 relative, the bar of the spectra), and the directional
derivative of every gradient against the oracle's central difference, which a quadratic
makes exact up to its rounding: 1e-12 of the loss over the step (2 h = 0.2 of the
direction), so 1e-9 of the loss; vsini at h = 1e-5, 1e-6 of the larger side."""
import numpy as np
import pytest

import oracle as O
from soap_gpu_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_phase,grid,map_res,n_mu,n,vsini,fac", [
    (1, 21, 9, 1, 2048, 2.0, False), (5, 40, 64, 6, 3001, 3.0, True), (10, 33, 17, 4, 2600, 0.05, True),
    (16, 24, 33, 3, 2500, 8.0, False), (17, 48, 16, 6, 2700, 2.0, True), (63, 16, 18, 2, 2300, 4.0, True),
    (65, 17, 31, 3, 2300, 1.0, False), (50, 30, 50, 10, 2311, 25.0, True)])
def test_diff_shapes(n_phase, grid, map_res, n_mu, n, vsini, fac):
    import torch
    from soap_gpu_amd.diff import DiffModel
    from soap_gpu_amd.engine import Engine, select_mask_lines
    rng = np.random.default_rng(n + n_phase)
    w = synth.small(seed=5, grid=grid, n=n, n_mu=n_mu, n_phase=1, n_lines=30, lmin=5000.0,
                    lmax=5000.0 * np.exp((n - 1) * 1e-6))
    sl, sw = select_mask_lines(w.wave, w.mask_l, w.mask_w, 210)
    lb = w.star["lb"]
    eng = Engine(0)
    model = DiffModel(eng, w.wave, w.mu_bounds, sl, sw, w.vgrid, grid, n_phase, map_res, w.sigma_inst, 210, lb=lb)
    q, s, f = (w.cubes[k] for k in ("q", "sp", "fac"))
    maps, fmaps = rng.uniform(0, 0.5, (n_phase, map_res, map_res)), rng.uniform(0, 0.5, (n_phase, map_res, map_res))
    target = 0.7 * grid * grid * (1.0 + 0.1 * rng.standard_normal((n_phase, n)))
    prm = np.array([vsini, 0.29, 0.34, 0.35] + ([1.15] if fac else []))
    z, ws = np.zeros(n_phase), 1.0 / float(np.sum(target[:, 210:-210] ** 2))

    def loss_of(prm, q, s, maps, f, fmaps):
        kf = prm[4] if fac else 0.0
        r = O.diff_forward(w.wave, grid, w.mu_bounds, *prm[:4], q, s, maps, w.sigma_inst, 210, w.vgrid, sl, sw, target,
                           z, z, w_spec=ws, w_rv=0.0, w_fw=0.0, kappa_f=kf, lb=lb, cube_f=f if fac else None,
                           fmaps=fmaps if fac else None)
        return r["loss"]

    def dev(a):
        return torch.tensor(a, dtype=torch.float64, device="cuda")

    args = [prm, q, s, maps, f, fmaps]
    got = model.forward(prm, dev(q), dev(s), dev(maps), dev(target), z, z, ws, 0.0, 0.0, f=dev(f) if fac else None,
                        fmaps=dev(fmaps) if fac else None)[0]
    ref = loss_of(*args)
    assert abs(got - ref) <= 1e-12 * abs(ref)
    g5, gq, gs, gm, gf, gfm = model.backward()
    grads = [g5[:len(prm)], gq.cpu().numpy(), gs.cpu().numpy(), gm.cpu().numpy()]
    grads += [gf.cpu().numpy(), gfm.cpu().numpy()] if fac else []
    for i, g in enumerate(grads):
        if i == 0:
            tries = [(np.eye(len(prm))[j], 0.1 if j else 1e-5) for j in range(len(prm))]
        else:
            tries = [(rng.uniform(0.0, 1.0, g.shape) * (args[i] if i in (1, 2, 4) else 0.3), 0.1)]
        for d, h in tries:
            fd = (loss_of(*args[:i], args[i] + h * d, *args[i + 1:])
                  - loss_of(*args[:i], args[i] - h * d, *args[i + 1:])) / (2 * h)
            an = float(np.sum(g * d))
            tol = 1e-9 * abs(ref) if h == 0.1 else 1e-6 * max(abs(fd), abs(ref))
            assert abs(an - fd) <= tol, (i, h, an, fd, ref)
    eng.close()
