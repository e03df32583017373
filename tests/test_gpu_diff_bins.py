"""The differentiable model when the mu bins are set anew between its calls: another
number of them is refused where buffers of the old number are bound or kept (a graph
step, a backward), and taken up by the next forward; going back to the bound number is
accepted again.  Other bins of the same number are taken up by the next forward and by the
next step, whether or not the step before it has been waited for."""
import numpy as np
import pytest

from soap_gpu_amd import synth
from soap_gpu_amd.engine import SoapError

pytestmark = pytest.mark.gpu

P, M, GRID = 3, 12, 40


def _problem(n_mu=4):
    import torch
    from soap_gpu_amd.diff import DiffModel
    from soap_gpu_amd.engine import Engine, select_mask_lines
    w = synth.small(seed=4, grid=GRID, n=2400, n_mu=n_mu, n_phase=1, n_lines=30, lmin=5000.0,
                    lmax=5000.0 * np.exp(2399 * 1e-6))
    sl, sw = select_mask_lines(w.wave, w.mask_l, w.mask_w, 210)
    rng = np.random.default_rng(8)
    dev = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")  # noqa: E731
    t = dict(prm=dev([2.0, 0.29, 0.34, 0.35, 1.15]), maps=dev(rng.uniform(0, 0.5, (P, M, M))),
             fmaps=dev(rng.uniform(0, 0.5, (P, M, M))), target=dev(900.0 + rng.standard_normal((P, w.n))),
             rv=dev(np.zeros(P)), fw=dev(np.full(P, 9e3)), bis=dev(np.zeros(P)),
             **{k: dev(w.cubes[c]) for k, c in (("q", "q"), ("s", "sp"), ("f", "fac"))})
    model = DiffModel(Engine(0), w.wave, w.mu_bounds, sl, sw, w.vgrid, GRID, P, M, w.sigma_inst, 210, lb=w.star["lb"])
    return w, model, t


WEIGHTS = (1e-6, 1e-3, 1e-5, 1e-3)


def _forward(model, t):
    return model.forward(t["prm"].cpu().numpy(), t["q"], t["s"], t["maps"], t["target"], np.zeros(P), np.full(P, 9e3),
                         *WEIGHTS[:3], bis_t=np.zeros(P), w_bis=WEIGHTS[3], f=t["f"], fmaps=t["fmaps"])[0]


def _bind(batch, t):
    import torch
    out = dict(loss=torch.zeros(1, dtype=torch.float64, device="cuda"), g5=torch.zeros_like(t["prm"]),
               gq=torch.zeros_like(t["q"]), gs=torch.zeros_like(t["q"]), gm=torch.zeros_like(t["maps"]),
               gf=torch.zeros_like(t["q"]), gfm=torch.zeros_like(t["maps"]))
    batch.bind(0, 9.0, t["prm"], t["q"], t["s"], t["maps"], t["target"], t["rv"], t["fw"], t["bis"], WEIGHTS,
               out["loss"], out["g5"], out["gq"], out["gs"], out["gm"], f=t["f"], fmaps=t["fmaps"], gf=out["gf"],
               gfm=out["gfm"])
    return out


@pytest.mark.parametrize("graph", [True, False])
def test_step_refuses_another_number_of_bins(graph):
    from soap_gpu_amd.diff import DiffBatch
    w, model, t = _problem()
    batch = DiffBatch([model])
    out = _bind(batch, t)
    batch.step(graph=graph)
    batch.sync()
    ref = {k: v.clone() for k, v in out.items()}
    for bounds in ([0.9, 0.7, 0.5, 0.3, 0.1], [0.5]):  # six bins, two bins
        model.eng.set_mu_bounds(np.array(bounds))
        with pytest.raises(SoapError, match="changed after binding"):
            batch.step(graph=graph)
    model.eng.set_mu_bounds(w.mu_bounds)
    for v in out.values():
        v.zero_()
    batch.step(graph=graph)
    batch.sync()
    for k, v in ref.items():
        assert bool((out[k] == v).all()), k
    batch.close()
    model.eng.close()


def test_backward_refuses_another_number_of_bins():
    w, model, t = _problem()
    loss = _forward(model, t)
    ref = model.backward()
    for bounds in ([0.9, 0.7, 0.5, 0.3, 0.1], [0.5]):
        model.eng.set_mu_bounds(np.array(bounds))
        with pytest.raises(SoapError, match="mu bins"):
            model.backward()
    model.eng.set_mu_bounds(w.mu_bounds)
    assert _forward(model, t) == loss
    for a, b in zip(model.backward(), ref):
        assert np.array_equal(np.asarray(a if isinstance(a, np.ndarray) else a.cpu()),
                              np.asarray(b if isinstance(b, np.ndarray) else b.cpu()))
    model.eng.close()


def _same_as_fresh(bounds, t, loss, grads):
    """Results against those of a new model on these bounds, bit for bit."""
    w, fresh, _ = _problem()
    fresh.eng.set_mu_bounds(bounds)
    assert _forward(fresh, t) == loss
    for a, b in zip(grads, fresh.backward()):
        a, b = (x if isinstance(x, np.ndarray) else x.cpu().numpy() for x in (a, b))
        np.testing.assert_array_equal(a, b)
    fresh.eng.close()


BOUNDS = [np.array(b) for b in ([0.95, 0.8, 0.2], [0.6, 0.4, 0.3], [0.75, 0.5, 0.25])]


def test_forward_takes_up_other_bins():
    w, model, t = _problem()
    _forward(model, t)
    for bounds in BOUNDS:
        model.eng.set_mu_bounds(bounds)
        loss = _forward(model, t)
        _same_as_fresh(bounds, t, loss, model.backward())
    model.eng.close()


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("wait", [True, False])
def test_step_takes_up_other_bins(graph, wait):
    import torch
    from soap_gpu_amd.diff import DiffBatch
    w, model, t = _problem()
    batch = DiffBatch([model])
    out = _bind(batch, t)
    torch.cuda.synchronize()
    batch.step(graph=graph)
    for bounds in BOUNDS:
        if wait:
            batch.sync()
        model.eng.set_mu_bounds(bounds)
        batch.step(graph=graph)
        batch.step(graph=graph)
    batch.sync()
    # a step's tap range is its bound vsini's, so its FIRs may add zeros that a forward leaves out
    got = [out["g5"], out["gq"], out["gs"], out["gm"], out["gf"], out["gfm"]]
    _same_as_fresh(BOUNDS[-1], t, float(out["loss"][0]), [x.cpu().numpy() for x in got])
    batch.close()
    model.eng.close()
