"""A structure's results do not depend on the batch around it: kernels that
choose another tile or launch shape by the batch's size give the same bits."""

import numpy as np
import pytest
import torch

from conftest import pkg, pkg_mod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,L,R_", [(128, 3, 20), (64, 2, 20), (32, 2, 16)])
def test_structures_alone_equal_the_batch(gpu, H, L, R_):
    """5,100 atoms in one batch (beyond the small-batch forms) against single
    structures of 1 to 300 atoms and a batch of 4,096 atoms exactly."""
    print(f"[case] batch invariance H{H}", flush=True)
    synth = pkg_mod("synth")
    rng = np.random.Generator(np.random.PCG64(7))
    sizes = [1, 2, 15, 16, 17, 31, 33, 104, 105, 300] + [64] * 54 + [16]
    sizes += [100] * 10
    mols = [synth.random_molecule(n, rng) for n in sizes]
    Z, P, ptr = synth.flatten(mols)
    torch.manual_seed(2)
    m = pkg().StudentForceField(hidden_dim=H, num_interactions=L, num_rbf=R_).to(gpu)
    Zt, Pt = torch.tensor(Z, device=gpu), torch.tensor(P.astype(np.float32), device=gpu)
    e, f, v = m.evaluate(Zt, Pt, np.array(sizes), need_virial=True)
    assert ptr[-1] > 4096 and ptr[65] == 4096
    for a, b in [(k, k + 1) for k in range(12)] + [(0, 65), (20, 36)]:
        s = slice(int(ptr[a]), int(ptr[b]))
        e1, f1, v1 = m.evaluate(Zt[s], Pt[s], np.array(sizes[a:b]), need_virial=True)
        assert torch.equal(f1, f[s]) and torch.equal(e1, e[a:b]) and torch.equal(v1, v[a:b]), a
