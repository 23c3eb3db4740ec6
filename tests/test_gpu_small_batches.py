"""Small batches: lists of at most 4096 atoms counted and filled in two launches,
message rows of at most 1024 atoms split over four sums.  Same bits as in a
larger batch."""
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


@pytest.mark.parametrize("sizes", [[1500, 1200], [4096], [63, 4033]])
def test_lists_up_to_4096_atoms(gpu, sizes):
    """Beside 4,097 single atoms the same structures take the general path."""
    print(f"[case] small list {sizes}", flush=True)
    synth = pkg_mod("synth")
    rng = np.random.Generator(np.random.PCG64(sum(sizes)))
    # atoms on a jittered grid, 2 A apart: a few dozen neighbours each
    def blob(n):
        k = int(np.ceil(n ** (1 / 3)))
        x = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
        return synth.Structure(np.full(n, 6), 2.0 * x + rng.uniform(-0.3, 0.3, (n, 3)))
    mols = [blob(n) for n in sizes]
    lone = [synth.Structure(np.array([6]), np.zeros((1, 3))) for _ in range(4097)]
    torch.manual_seed(3)
    m = pkg().StudentForceField(hidden_dim=32, num_interactions=1, num_rbf=8,
                                cutoff=3.5).to(gpu)

    def run(ms):
        Z, P, ptr = synth.flatten(ms)
        return m.evaluate(torch.tensor(Z, device=gpu),
                          torch.tensor(P.astype(np.float32), device=gpu), np.diff(ptr),
                          need_virial=True)

    e, f, v = run(mols)
    e2, f2, v2 = run(mols + lone)
    n, B = sum(sizes), len(sizes)
    assert torch.equal(e, e2[:B]) and torch.equal(f, f2[:n]) and torch.equal(v, v2[:B])


@pytest.mark.parametrize("n_side", [5, 11])
def test_cell_list_in_one_workgroup(gpu, n_side, monkeypatch):
    """A water box with the cell list against the brute-force image search: one
    below and one near the bound of the single-workgroup build (3,993 atoms)."""
    print(f"[case] cell list {n_side}", flush=True)
    synth, engine = pkg_mod("synth"), pkg_mod("engine")
    box = synth.water_box(n_side, seed=1)
    cell = np.asarray(box.cell, dtype=np.float64).reshape(3, 3)
    Z = torch.tensor(box.numbers, device=gpu)
    x = torch.tensor(box.positions.astype(np.float32), device=gpu)
    torch.manual_seed(4)
    kw = dict(hidden_dim=32, num_interactions=1, num_rbf=8, cutoff=4.0)
    m = pkg().StudentForceField(**kw).to(gpu)
    got = m.energy_forces_virial(Z, x, cell, np.ones(3, bool))
    monkeypatch.setattr(engine, "CELL_LIST_MIN_ATOMS", 1 << 30)
    m2 = pkg().StudentForceField(**kw).to(gpu)
    m2.load_state_dict(m.state_dict())
    for a, b in zip(got, m2.energy_forces_virial(Z, x, cell, np.ones(3, bool))):
        assert torch.equal(a, b)
