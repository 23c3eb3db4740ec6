"""Batches of at most 1024 atoms: lists counted and filled in two launches, rows
of the messages split over four sums.  Same bits as in a larger batch."""
import numpy as np
import pytest
import torch

from conftest import pkg, pkg_mod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [128, 64, 32])
@pytest.mark.parametrize("sizes", [[1], [2, 63], [64], [65, 1], [5, 129], [200, 1, 320],
                                   [1, 1023], [1024]])
def test_small_batch_equals_larger_batch(gpu, sizes, H):
    """Every word edge of a row's hit mask, with structures that start anywhere;
    beside 1,025 single atoms the same structures take the general path."""
    print(f"[case] small batch {sizes} H{H}", flush=True)
    synth = pkg_mod("synth")
    rng = np.random.Generator(np.random.PCG64(sum(sizes)))
    mols = [synth.random_molecule(n, rng) for n in sizes]
    lone = [synth.random_molecule(1, rng) for _ in range(1025)]
    torch.manual_seed(3)
    m = pkg().StudentForceField(hidden_dim=H, num_interactions=2, num_rbf=20).to(gpu)

    def run(ms):
        Z, P, ptr = synth.flatten(ms)
        return m.evaluate(torch.tensor(Z, device=gpu),
                          torch.tensor(P.astype(np.float32), device=gpu),
                          np.array([len(z) for z in np.split(Z, ptr[1:-1])]), need_virial=True)

    e, f, v = run(mols)
    e2, f2, v2 = run(mols + lone)
    n, B = sum(sizes), len(sizes)
    assert torch.equal(e, e2[:B]) and torch.equal(f, f2[:n]) and torch.equal(v, v2[:B])
