"""A gradient with respect to the positions alone does no parameter pass, and
every other call gets the same gradients as before."""
import numpy as np
import pytest
import torch

from conftest import pkg, pkg_mod

pytestmark = pytest.mark.gpu


def test_parameter_pass_runs_only_where_it_is_asked_for(gpu, monkeypatch):
    print("[case] parameter pass on demand", flush=True)
    train, synth = pkg_mod("train"), pkg_mod("synth")
    rng = np.random.Generator(np.random.PCG64(3))
    Z, P, _ = synth.flatten([synth.random_molecule(9, rng)])
    torch.manual_seed(0)
    m = pkg().StudentForceField(hidden_dim=32, num_interactions=2).to(gpu)
    Zt = torch.tensor(Z, device=gpu)
    x = torch.tensor(P.astype(np.float32), device=gpu).requires_grad_(True)
    calls = []
    real = train.reverse

    def counted(*a, **k):
        calls.append(k.get("lam") is not None)
        return real(*a, **k)
    monkeypatch.setattr(train, "reverse", counted)
    params = list(m.parameters())
    E = m(Zt, x)
    (g,) = torch.autograd.grad(E, x, create_graph=True)
    assert calls == []
    # through the gradient, to one parameter and to all
    w = m.interactions[0].update.update_mlp[0].weight
    (gw,) = torch.autograd.grad((g ** 2).sum(), w, retain_graph=True)
    assert calls == [True]
    (gw1,) = torch.autograd.grad(E, w, retain_graph=True)
    assert calls == [True, False]
    both = torch.autograd.grad(E, [x] + params, retain_graph=True)
    assert calls == [True, False, False]
    k = [p is w for p in params].index(True)
    assert torch.equal(both[1 + k], gw1) and torch.equal(both[0], g.detach())
    (E + (g ** 2).sum()).backward()
    assert sorted(calls[3:]) == [False, True]   # one pass each, in either order
    assert torch.allclose(w.grad, gw + gw1, rtol=0, atol=1e-6 * (gw.abs().max() + gw1.abs().max()))
