"""The filter's distance tables (csrc/filter_table.hip) on the GPU: distances
at and around the knots and the cutoff, weights that the tables cannot follow,
and the evaluations right after a weight change, against the FP64 oracle."""

import numpy as np
import pytest
import torch

from conftest import pkg, pkg_mod
from oracle import painn_ref as R

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[case] {msg}", flush=True)


def _model(H, L, R_, rc, bias=0.05):
    torch.manual_seed(0)
    m = pkg().StudentForceField(hidden_dim=H, num_interactions=L, num_rbf=R_, cutoff=rc)
    with torch.no_grad():
        for n, p in m.named_parameters():
            if n.endswith(".bias"):
                p.copy_(bias * torch.randn(p.shape))
    return m.to("cuda:0")


def _check(model, Z, P32, sizes, rc):
    """Energies and forces against FP64: within three times what the same
    algorithm's float32 on the CPU is off, plus 1e-6 of the largest value (the
    float32 rounding of sums over a few neighbours)."""
    e, f, _ = model.evaluate(torch.tensor(Z, device="cuda:0"), torch.tensor(P32, device="cuda:0"),
                             np.asarray(sizes))
    sd = {k: v.detach().cpu() for k, v in model.state_dict().items()}
    b = np.repeat(np.arange(len(sizes)), sizes)
    E, F = R.energy_and_forces(sd, Z, P32.astype(np.float64), rc, batch=b, n_structures=len(sizes))
    E32, F32 = R.energy_and_forces(sd, Z, P32, rc, batch=b, n_structures=len(sizes),
                                   dtype=torch.float32)
    for got, want, ref in ((e.cpu(), E, E32), (f.cpu().double(), F, F32)):
        tol = 3.0 * (ref.double() - want).abs().max() + 1e-6 * want.abs().max()
        assert (got - want).abs().max() <= tol, ((got - want).abs().max(), tol)
    return e, f


@pytest.mark.parametrize("H,R_,rc", [(32, 16, 5.0), (64, 1, 5.0), (128, 20, 4.7), (64, 32, 6.0)])
def test_dimers_at_knots_and_cutoff(gpu, H, R_, rc):
    """Dimers along x (the distance is the float32 coordinate itself): at the
    first and last knots, one ulp either side of knots, in the middle of
    intervals, nearly coincident and within a few ulp of the cutoff."""
    note(f"table dimers H{H} R{R_} rc {rc}")
    h = np.float32(2.0 ** -9)
    d = [h, 2 * h, 3 * h, np.float32(0.5) * h, np.float32(1e-4)]
    for k in (0.5, 1.0, 1.25, 2.0, 3.0 + h):
        x = np.float32(k)
        d += [x, np.nextafter(x, np.float32(0)), np.nextafter(x, np.float32(9)), x + h / 2]
    c = np.float32(rc)
    for _ in range(3):
        d.append(c)
        c = np.nextafter(c, np.float32(0))
    d += [np.float32(rc) - h, np.float32(rc) - h / 2, np.float32(rc) + h]
    P = np.zeros((2 * len(d), 3), dtype=np.float32)
    P[1::2, 0] = d
    Z = np.tile([6, 1], len(d))
    _check(_model(H, 2, R_, rc), Z, P, [2] * len(d), rc)


@pytest.mark.parametrize("what", ["narrow", "steep", "one narrow"])
def test_weights_beyond_the_tables(gpu, what):
    """Basis widths below the knot spacing, or a first layer so steep that the
    filter turns within an interval: the guard keeps the direct product."""
    note(f"table guard: {what}")
    m = _model(64, 2, 20, 5.0)
    with torch.no_grad():
        if what == "narrow":
            m.rbf.widths.fill_(2.0 ** -10)
        elif what == "one narrow":
            m.rbf.widths[7] = 0.004
        else:
            m.interactions[1].message.rbf_to_scalar[0].weight.mul_(3e3)
    mols = pkg_mod("synth").molecule_set(6, 5, 30, seed=9)
    Z, P, ptr = pkg_mod("synth").flatten(mols)
    _check(m, Z, P.astype(np.float32), np.diff(ptr), 5.0)


@pytest.mark.parametrize("narrow", [False, True])
def test_evaluations_after_a_weight_change(gpu, narrow):
    """The first evaluation after a weight change launches both forms behind
    the guard's flag, the next one the chosen form: same bits, and those of a
    plan that was bound to the new weights."""
    note(f"table refresh, narrow {narrow}")
    m = _model(32, 2, 16, 5.0)
    mols = pkg_mod("synth").molecule_set(5, 5, 40, seed=3)
    Z, P, ptr = pkg_mod("synth").flatten(mols)
    P32, sizes = P.astype(np.float32), np.diff(ptr)
    before = _check(m, Z, P32, sizes, 5.0)
    with torch.no_grad():
        m.interactions[0].message.rbf_to_scalar[2].weight.mul_(1.1)
        if narrow:
            m.rbf.widths.mul_(0.02)
    runs = [_check(m, Z, P32, sizes, 5.0) for _ in range(3)]
    m._plans.clear()
    runs.append(_check(m, Z, P32, sizes, 5.0))
    assert not torch.equal(before[1], runs[0][1])
    for e, f in runs[1:]:
        assert torch.equal(e, runs[0][0]) and torch.equal(f, runs[0][1])


@pytest.mark.parametrize("H,n", [(32, 40), (64, 40), (128, 40), (128, 400)])
def test_first_block_without_its_zero_vectors(gpu, H, n):
    """The first evaluation with new weights runs before its tables are checked
    and multiplies the first block's zero vectors out; the ones after leave them
    out (row forms of up to and beyond 1,024 atoms).  The same bits; a NaN in the
    filter rows that only they meet still reaches the energy."""
    print(f"[case] first block H{H} n{n}", flush=True)
    synth = pkg_mod("synth")
    rng = np.random.Generator(np.random.PCG64(n))
    Z, P, ptr = synth.flatten([synth.random_molecule(40, rng) for _ in range(n // 10)])
    torch.manual_seed(1)
    m = pkg().StudentForceField(hidden_dim=H, num_interactions=2, num_rbf=20).to(gpu)
    Zt, Pt = torch.tensor(Z, device=gpu), torch.tensor(P.astype(np.float32), device=gpu)
    sizes = np.diff(ptr)
    ev = lambda: m.evaluate(Zt, Pt, sizes, need_virial=True)
    for a in (ev(), ev()):     # resolve the tables
        assert torch.isfinite(a[0]).all()
    with torch.no_grad():
        m.interactions[0].message.rbf_to_scalar[2].weight.mul_(1.0)
    runs = [ev() for _ in range(4)]
    for r in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(runs[0], r))
    with torch.no_grad():
        m.interactions[0].message.rbf_to_scalar[2].weight[H + 3, 5] = float("nan")
    for _ in range(4):
        assert torch.isnan(ev()[0]).all()


@pytest.mark.parametrize("H,n", [(32, 8), (64, 70), (128, 30), (128, 141)])
def test_runs_of_pairs_keep_a_structures_bits(gpu, H, n):
    """The filter adjoint takes one, two or four pairs per group of lanes with the
    batch's size; an atom's run of pairs ends anywhere in them.  A structure gives
    the bits it gives alone (one pair per group)."""
    print(f"[case] pair runs H{H} n{n}", flush=True)
    synth = pkg_mod("synth")
    rng = np.random.Generator(np.random.PCG64(n))
    Z, P, ptr = synth.flatten([synth.random_molecule(41 + k % 20, rng) for k in range(n)])
    torch.manual_seed(1)
    m = pkg().StudentForceField(hidden_dim=H, num_interactions=3, num_rbf=20, cutoff=8.0).to(gpu)
    Zt, Pt = torch.tensor(Z, device=gpu), torch.tensor(P.astype(np.float32), device=gpu)
    for _ in range(3):         # resolve the tables
        e, f, v = m.evaluate(Zt, Pt, np.diff(ptr), need_virial=True)
    for k in (0, n // 2, n - 1):
        at = slice(int(ptr[k]), int(ptr[k + 1]))
        for _ in range(3):
            one = m.evaluate(Zt[at], Pt[at], np.diff(ptr)[k:k + 1], need_virial=True)
        assert torch.equal(one[0][0], e[k]) and torch.equal(one[1], f[at])
        assert torch.equal(one[2][0], v[k])


@pytest.mark.parametrize("H", [32, 64, 128])
@pytest.mark.parametrize("L", [1, 2])
def test_last_block_without_its_vectors(gpu, H, L):
    """The last block's update forms its scalars only: against the float64 model for
    few atoms, and a structure's bits in the forms of up to 1,024, up to 4,096 and
    more atoms."""
    print(f"[case] last block H{H} L{L}", flush=True)
    synth = pkg_mod("synth")
    rng = np.random.Generator(np.random.PCG64(H + L))
    Z, P, ptr = synth.flatten([synth.random_molecule(41, rng) for _ in range(110)])
    torch.manual_seed(1)
    m = pkg().StudentForceField(hidden_dim=H, num_interactions=L, num_rbf=20).to(gpu)
    P32, sizes = P.astype(np.float32), np.diff(ptr)
    n = int(ptr[3])
    _check(m, Z[:n], P32[:n], sizes[:3], 5.0)
    Zt, Pt = torch.tensor(Z, device=gpu), torch.tensor(P32, device=gpu)
    runs = []
    for k in (3, 40, 110):
        for _ in range(3):     # resolve the tables
            r = m.evaluate(Zt[:ptr[k]], Pt[:ptr[k]], sizes[:k], need_virial=True)
        runs.append((r[0][:3], r[1][:n], r[2][:3]))
    for r in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(runs[0], r))


def _plans(blobs, H=64, L=2, R_=20):
    """A batch, and for every weight blob the results of a plan bound to it."""
    synth, engine = pkg_mod("synth"), pkg_mod("engine")
    dev = torch.device("cuda:0")
    Z, P, ptr = synth.flatten(synth.molecule_set(5, 10, 40, seed=4))
    pos = torch.tensor(P.astype(np.float32), device=dev)
    lay = engine.make_layout(np.diff(ptr), dev)
    numbers = torch.tensor(Z, dtype=torch.int64, device=dev)
    cap = engine.edge_capacity_bound(np.diff(ptr), False)
    new = lambda w: engine.Plan(H, L, R_, 118, 5.0, lay, numbers, w, cap)
    outs = lambda: (torch.empty(len(ptr) - 1, dtype=torch.float64, device=dev),
                    torch.empty(len(Z), 3, dtype=torch.float32, device=dev))

    def run(plan):
        o = outs()
        plan.energy_forces(pos, *o)
        return o
    return pos, new, outs, run, [run(new(w)) for w in blobs]


def _blobs():
    """Two sets of weights that the tables follow and one that they cannot."""
    models = [_model(64, 2, 20, 5.0, bias) for bias in (0.05, 0.3, 0.3)]
    with torch.no_grad():
        models[2].rbf.widths.mul_(0.02)
    return [m.packed_weights("cuda:0") for m in models]


def _equal(a, b):
    assert all(torch.equal(x, y) for x, y in zip(a, b))


def _captured(plan, pos, o):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.energy_forces(pos, *o)
    return g


@pytest.mark.parametrize("new", [1, 2])
def test_capture_right_after_a_weight_change(gpu, new):
    """New weights, a capture, then eager evaluations before and between the
    graph's replays: all with the new weights, and after another change too."""
    note(f"capture after set_weights, blob {new}")
    blobs = _blobs()
    pos, make, outs, run, want = _plans(blobs)
    plan = make(blobs[0])
    for _ in range(3):
        _equal(run(plan), want[0])
    plan.set_weights(blobs[new])
    o = outs()
    g = _captured(plan, pos, o)
    _equal(run(plan), want[new])
    for _ in range(3):
        for t in o:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        _equal(o, want[new])
        _equal(run(plan), want[new])
    plan.set_weights(blobs[0])
    for _ in range(3):
        _equal(run(plan), want[0])


def test_replays_follow_weights_written_in_place(gpu):
    """A captured evaluation, its blob rewritten and bound again: replays and eager
    evaluations give the new weights' results, with tables and without."""
    note("replays after in-place weight changes")
    blobs = _blobs()
    pos, make, outs, run, want = _plans(blobs)
    w = blobs[0].clone()
    plan = make(w)
    for _ in range(3):
        _equal(run(plan), want[0])
    o = outs()
    g = _captured(plan, pos, o)
    for k in (0, 1, 2, 1, 2, 0):
        w.copy_(blobs[k])
        plan.set_weights(w)
        for _ in range(2):
            for t in o:
                t.zero_()
            g.replay()
            torch.cuda.synchronize()
            _equal(o, want[k])
            _equal(run(plan), want[k])


def test_weights_bound_inside_a_capture(gpu):
    """set_weights and an evaluation in one graph: every replay takes the blob as it
    is then, and eager evaluations follow what the last replay bound."""
    note("set_weights inside a capture")
    blobs = _blobs()
    pos, make, outs, run, want = _plans(blobs)
    w = blobs[0].clone()
    plan = make(w)
    run(plan)
    o = outs()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.set_weights(w)
        plan.energy_forces(pos, *o)
    for k in (0, 1, 2, 1, 0):
        w.copy_(blobs[k])
        g.replay()
        torch.cuda.synchronize()
        _equal(o, want[k])
        for _ in range(3):
            _equal(run(plan), want[k])


def test_evaluations_beside_a_capture_of_another_stream(gpu):
    """While one stream is being captured, evaluations on another one run (the
    second one after a weight change is the one that reads the tables' flag)."""
    note("evaluations beside a capture")
    blobs = _blobs()
    pos, make, outs, run, want = _plans(blobs)
    plan, side = make(blobs[0]), torch.cuda.Stream()
    x = torch.zeros(64, device=gpu)
    plan.set_weights(blobs[1])
    o = [outs() for _ in range(3)]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        x.add_(1.0)
        for q in o:
            plan.energy_forces(pos, *q, stream=side)
    g.replay()
    torch.cuda.synchronize()
    assert float(x[0]) == 1.0
    for q in o:
        _equal(q, want[1])


def test_stage_of_the_first_blocks_message_adjoint(gpu, monkeypatch):
    """Block 0's message adjoint as a stage reads filter columns that the evaluation
    itself does not need: in a workspace of NaN bytes, what the stage writes is
    finite, and the same twice."""
    note("stage: message adjoint of block 0")
    engine, C = pkg_mod("engine"), pkg_mod("_capi")
    empty = torch.empty
    monkeypatch.setattr(engine.torch, "empty",
                        lambda *a, **k: empty(*a, **k).fill_(255) if k.get("dtype") == torch.uint8
                        else empty(*a, **k))
    pos, make, outs, run, want = _plans([_model(64, 2, 20, 5.0).packed_weights("cuda:0")])
    plan = make(_model(64, 2, 20, 5.0).packed_weights("cuda:0"))
    for _ in range(3):
        _equal(run(plan), want[0])
    written = []
    before = plan.workspace.view(torch.int32).clone()
    for _ in range(2):
        C.check("stage", C.lib().mlff_launch_stage(plan.handle, C.stream_handle(), 7, 0))
        after = plan.workspace.view(torch.int32).clone()
        new = after != before
        assert new.any() and torch.isfinite(after[new].view(torch.float32)).all()
        written.append(after)
    assert torch.equal(*written)


@pytest.mark.parametrize("n,ecap", [(2000, 100000), (2000, 3), (4200, 400000)])
def test_long_rows_cut_off_by_the_edge_capacity(gpu, monkeypatch, n, ecap):
    """Rows of more than 256 neighbours from the cell list, more edges than their
    capacity and room for every pair: the pairs of the rows that are cut off are read
    by the pair kernels.  In a workspace of NaN bytes the overflow is flagged and the
    results are finite; with the capacity that the counters ask for they are those
    of a plan that was large enough."""
    note(f"long rows cut off, {n} atoms, {ecap} edges")
    engine, C = pkg_mod("engine"), pkg_mod("_capi")
    empty = torch.empty
    monkeypatch.setattr(engine.torch, "empty",
                        lambda *a, **k: empty(*a, **k).fill_(255) if k.get("dtype") == torch.uint8
                        else empty(*a, **k))
    dev = torch.device("cuda:0")
    rng = np.random.Generator(np.random.PCG64(n))
    box = 15.1 * (n / 2000) ** (1 / 3)
    pos = torch.tensor((rng.random((n, 3)) * box).astype(np.float32), device=dev)
    lay = engine.make_layout([n], dev, np.eye(3)[None] * box, np.ones((1, 3)))
    numbers = torch.ones(n, dtype=torch.int64, device=dev)
    m = _model(32, 1, 16, 5.0)
    edges = engine.count_edges(pos, lay, 5.0)
    assert edges > 256 * n

    def run(cap):
        plan = engine.Plan(32, 1, 16, m.max_z, 5.0, lay, numbers, m.packed_weights(dev), cap,
                           pair_capacity=edges // 2 + 64)
        assert plan.cell_grid[0, 0] >= 3
        o = (empty(1, dtype=torch.float64, device=dev), empty(n, 3, device=dev))
        for _ in range(2):
            plan.energy_forces(pos, *o)
        c = plan.read_counts()
        assert c[C.MLFF_COUNT_EDGES] == edges and bool(c[C.MLFF_COUNT_OVERFLOW]) == (cap < edges)
        assert all(torch.isfinite(t).all() for t in o)
        return o

    run(ecap)
    a, b = run(edges), run(edges + 1000)
    _equal(a, b)


@pytest.mark.parametrize("narrow,n", [(False, 3), (False, 40), (True, 3), (True, 40)])
def test_tuner_leaves_shapes_alone_that_nothing_reads(gpu, narrow, n):
    """With tables the direct filter kernels do not run, up to 1,024 atoms the message
    rows take one form: the tuner times the kinds that are read, and the others keep
    their defaults.  Same bits after it."""
    note(f"tuner, narrow {narrow}, {n} molecules")
    synth, engine, tuner = pkg_mod("synth"), pkg_mod("engine"), pkg_mod("autotune")
    dev = torch.device("cuda:0")
    Z, P, ptr = synth.flatten(synth.molecule_set(n, 30, 50, seed=n))
    pos = torch.tensor(P.astype(np.float32), device=dev)
    lay = engine.make_layout(np.diff(ptr), dev)
    m = _model(64, 2, 20, 5.0)
    if narrow:
        with torch.no_grad():
            m.rbf.widths.mul_(0.02)
    plan = engine.Plan(64, 2, 20, 118, 5.0, lay, torch.tensor(Z, device=dev),
                       m.packed_weights(dev), engine.edge_capacity_bound(np.diff(ptr), False))
    o = (torch.empty(n, dtype=torch.float64, device=dev), torch.empty(len(Z), 3, device=dev))
    plan.energy_forces(pos, *o)
    before = [t.clone() for t in o]
    tuner._CACHE.clear()
    got = tuner.tune(plan, pos, candidates=[512], reps=2)
    used = {k: (narrow if k.startswith("filter") else len(Z) > 1024) for k in tuner.SHAPE_NAMES}
    assert plan.shapes_used() == tuple(used[k] for k in tuner.SHAPE_NAMES)
    timed = {k.split("=")[0] for k in got["shape_timings_us"]} - {"default"}
    assert timed <= {k for k in used if used[k]} and (not any(used.values()) or timed)
    for k, shape, default in zip(tuner.SHAPE_NAMES, got["tiles"], engine.default_tiles(64)):
        assert used[k] or shape == default
    plan.energy_forces(pos, *o)
    _equal(o, before)
