"""Interaction blocks on a caller-given edge list: the grouping kernels and the
blocks' own autograd functions against torch's sort and the module path."""
import pytest
import torch

from conftest import pkg_mod
from oracle import painn_ref as R_

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[0, 1, 0], [64, 65, 63, 0], [2048, 2049, 5], [300] * 40, [1]])
def test_edge_groups_equal_a_stable_sort(gpu, sizes):
    """Every row form (registers, ranking, scan), empty rows, duplicate edges."""
    print(f"[case] edge groups {sizes[:4]}", flush=True)
    model = pkg_mod("model")
    n = len(sizes)
    gen = torch.Generator().manual_seed(1)
    dst = torch.repeat_interleave(torch.arange(n), torch.tensor(sizes))
    dst = dst[torch.randperm(len(dst), generator=gen)].to(gpu)
    src = torch.randint(0, n, (len(dst),), generator=gen).to(gpu)
    row_ptr, col, eid, ends = model._edge_csr(src, dst, n, 2)
    assert torch.equal(ends[0].long(), dst) and torch.equal(ends[1].long(), src)
    for l, (key, other) in enumerate(((dst, src), (src, dst))):
        order = torch.sort(key, stable=True).indices
        assert torch.equal(eid[l].long(), order) and torch.equal(col[l].long(), other[order])
        assert torch.equal(row_ptr[l, 1:].long(), torch.cumsum(torch.bincount(key, minlength=n), 0))


@pytest.mark.parametrize("bad", [-1, 5])
def test_edges_out_of_range_are_refused(gpu, bad):
    print(f"[case] edge out of range {bad}", flush=True)
    model = pkg_mod("model")
    ok = torch.tensor([0, 1, 2], device=gpu)
    for src, dst in ((torch.tensor([0, bad, 1], device=gpu), ok),
                     (ok, torch.tensor([0, 1, bad], device=gpu))):
        with pytest.raises(ValueError, match="outside"):
            model._edge_csr(src, dst, 5, 2)


@pytest.mark.parametrize("H,R,n,E", [(64, 20, 50, 3000), (32, 9, 3, 1), (128, 32, 70, 2049)])
def test_blocks_equal_the_module_path(gpu, H, R, n, E):
    """A forward hook takes the module path.  Outputs, gradients and gradients of
    a gradient norm agree to 2e-5 of their norm: sums of up to 3,000 float32
    products have an error of about sqrt(3000) 2^-24 = 3.3e-6."""
    print(f"[case] blocks H{H} R{R} n{n} E{E}", flush=True)
    model = pkg_mod("model")
    torch.manual_seed(5)
    blk = model.PaiNNInteraction(H, R).to(gpu)
    ins = [torch.randn(*sh, device=gpu).requires_grad_(True)
           for sh in ((n, H), (n, 3, H), (E, R), (E, 3))]
    edges = torch.randint(0, n, (2, E), device=gpu)
    leaves = ins + list(blk.parameters())
    gs, gv = torch.randn(n, H, device=gpu), torch.randn(n, 3, H, device=gpu)

    def run():
        out = blk(ins[0], ins[1], edges, ins[2], ins[3])
        first = torch.autograd.grad(out, leaves, (gs, gv), retain_graph=True)
        s, v = blk.update(ins[0], ins[1])
        g = torch.autograd.grad((s * gs).sum() + (v * gv).sum(), ins[:2], create_graph=True)
        second = torch.autograd.grad(sum((t ** 2).sum() for t in g),
                                     ins[:2] + list(blk.update.parameters()))
        return list(out) + list(first) + list(second)

    fused = run()
    names = [type(t.grad_fn).__name__ for t in blk.update(ins[0], ins[1])]
    assert names[0].startswith("_UpdateBlock")
    for seq in (blk.message.rbf_to_scalar, blk.update.update_mlp):
        seq.register_forward_hook(lambda *a: None)
    plain = run()
    assert not type(blk.update(ins[0], ins[1])[0].grad_fn).__name__.startswith("_UpdateBlock")
    for k, (a, b) in enumerate(zip(fused, plain)):
        assert (a - b).norm() <= 2e-5 * b.norm() + 1e-30, k


def test_blocks_take_a_strided_edge_list(gpu):
    """The rows of an [E, 2] list's transpose are strided: the lists, outputs and
    gradients of the contiguous edge list, bit for bit."""
    print("[case] strided edge list", flush=True)
    model = pkg_mod("model")
    gen = torch.Generator().manual_seed(2)
    H, R, n, E = 64, 20, 50, 3000
    pairs = torch.randint(0, n, (E, 2), generator=gen).to(gpu)
    torch.manual_seed(3)
    blk = model.PaiNNInteraction(H, R).to(gpu)
    ins = [torch.randn(*sh, generator=gen).to(gpu).requires_grad_(True)
           for sh in ((n, H), (n, 3, H), (E, R), (E, 3))]

    def run(edges):
        out = blk(ins[0], ins[1], edges, ins[2], ins[3])
        grads = torch.autograd.grad(out[0].square().sum() + out[1].square().sum(),
                                    ins + list(blk.parameters()))
        return list(model._edge_csr(edges[0], edges[1], n, 2)) + list(out) + list(grads)

    assert not pairs.t()[0].is_contiguous()
    for k, (a, b) in enumerate(zip(run(pairs.t()), run(pairs.t().contiguous()))):
        assert torch.equal(a, b), k


@pytest.mark.parametrize("H,K", [(32, 64), (64, 256), (64, 32), (128, 16)])
def test_layers_of_another_width_take_the_module_path(gpu, H, K):
    """update_mlp and rbf_to_scalar with K hidden channels: the block's outputs and
    gradients in float64 (2e-5 of the norm, as above)."""
    print(f"[case] other widths H{H} K{K}", flush=True)
    nn, model = torch.nn, pkg_mod("model")
    torch.manual_seed(7)
    n, E, R = 30, 400, 12
    blk = model.PaiNNInteraction(H, R).to(gpu)
    blk.update.update_mlp = nn.Sequential(nn.Linear(2 * H, K), nn.SiLU(), nn.Linear(K, 3 * H)).to(gpu)
    blk.message.rbf_to_scalar = nn.Sequential(nn.Linear(R, K), nn.SiLU(),
                                              nn.Linear(K, 3 * H)).to(gpu)
    ins = [torch.randn(*sh, device=gpu).requires_grad_(True)
           for sh in ((n, H), (n, 3, H), (E, R), (E, 3))]
    edges = torch.randint(0, n, (2, E), device=gpu)
    leaves = ins + list(blk.parameters())
    out = blk(ins[0], ins[1], edges, ins[2], ins[3])
    got = list(out) + list(torch.autograd.grad(out[0].square().sum() + out[1].square().sum(), leaves))
    sd = {f"interactions.0.{k}": p.detach().cpu().double().requires_grad_(True)
          for k, p in blk.named_parameters()}
    s, v, rbf, ev = rins = [t.detach().cpu().double().requires_grad_(True) for t in ins]
    ei = edges.cpu()
    want = R_.update(sd, 0, H, *R_.message(sd, 0, H, s, v, ei[0], ei[1], rbf, ev))
    want = list(want) + list(torch.autograd.grad(
        want[0].square().sum() + want[1].square().sum(), rins + list(sd.values())))
    for k, (a, b) in enumerate(zip(got, want)):
        assert (a.detach().cpu().double() - b.detach()).norm() <= 2e-5 * b.norm() + 1e-30, k


def test_an_update_of_the_wrong_output_width_is_refused(gpu):
    print("[case] wrong output width", flush=True)
    nn, model = torch.nn, pkg_mod("model")
    blk = model.PaiNNUpdate(64).to(gpu)
    blk.update_mlp[2] = nn.Linear(64, 256).to(gpu)
    with pytest.raises(RuntimeError):
        blk(torch.randn(5, 64, device=gpu), torch.randn(5, 3, 64, device=gpu))


def test_second_derivatives_where_one_input_depends_on_another(gpu):
    """v = f(s), and a bias that s was formed from: the gradient of a gradient norm
    equals the module path's (2e-5 of the norm, as above)."""
    print("[case] dependent inputs, second derivatives", flush=True)
    model = pkg_mod("model")
    torch.manual_seed(8)
    n, H, E, R = 20, 64, 200, 12
    upd, msg = model.PaiNNUpdate(H).to(gpu), model.PaiNNMessage(H, R).to(gpu)
    x = torch.randn(n, H, device=gpu).requires_grad_(True)
    y = torch.randn(E, R, device=gpu).requires_grad_(True)

    def run(apply):
        s = x * torch.sigmoid(upd.update_mlp[0].bias)
        v = torch.stack([s.sin(), s.cos(), s * s], dim=1)
        so, vo = upd(s, v)
        w = msg.rbf_to_scalar
        x2 = y * w[2].bias[:R]
        filt = apply(x2, w[0].weight, w[0].bias, w[2].weight, w[2].bias)
        leaves = [x, y] + list(upd.parameters()) + list(w.parameters())
        g = torch.autograd.grad(so.square().sum() + vo.square().sum() + filt.square().sum(), leaves,
                                create_graph=True)
        return list(g) + list(torch.autograd.grad(sum(t.square().sum() for t in g), leaves))

    fused = run(model._EdgeFilter.apply)
    upd.update_mlp.register_forward_hook(lambda *a: None)
    plain = run(lambda t, *w: msg.rbf_to_scalar(t))
    for k, (a, b) in enumerate(zip(fused, plain)):
        assert (a - b).norm() <= 2e-5 * b.norm() + 1e-30, k


def test_batched_gradients(gpu):
    """is_grads_batched and vectorized Jacobians, one gradient after the other."""
    print("[case] batched gradients", flush=True)
    model = pkg_mod("model")
    torch.manual_seed(9)
    n, H, R = 7, 32, 12
    upd, mlp = model.PaiNNUpdate(H).to(gpu), model.PaiNNMessage(H, R).to(gpu).rbf_to_scalar
    s = torch.randn(n, H, device=gpu).requires_grad_(True)
    v = torch.randn(n, 3, H, device=gpu).requires_grad_(True)
    x = torch.randn(n, R, device=gpu).requires_grad_(True)
    filt = model._EdgeFilter.apply(x, mlp[0].weight, mlp[0].bias, mlp[2].weight, mlp[2].bias)
    for out, leaves in ((upd(s, v), [s, v] + list(upd.parameters())),
                        ((filt,), [x] + list(mlp.parameters()))):
        gs = [torch.randn(4, *t.shape, device=gpu) for t in out]
        got = torch.autograd.grad(out, leaves, gs, is_grads_batched=True, retain_graph=True)
        for k in range(4):
            one = torch.autograd.grad(out, leaves, [g[k] for g in gs], retain_graph=True)
            for q, (a, b) in enumerate(zip(got, one)):
                assert (a[k] - b).norm() <= 2e-5 * b.norm() + 1e-30, (k, q)


@pytest.mark.parametrize("whole", [True, False])
def test_captured_update_block(gpu, whole):
    """The update block's forward and backward, or its backward alone, in a graph:
    every replay gives the eager gradients of the inputs as they are then (2e-5 of
    the norm, as above), with other work and other pinned memory in between."""
    print(f"[case] captured update block, forward too: {whole}", flush=True)
    model = pkg_mod("model")
    torch.manual_seed(10)
    n, H = 16, 64
    upd = model.PaiNNUpdate(H).to(gpu)
    s = torch.randn(n, H, device=gpu).requires_grad_(True)
    v = torch.randn(n, 3, H, device=gpu).requires_grad_(True)
    gs = [torch.randn(n, H, device=gpu), torch.randn(n, 3, H, device=gpu)]
    leaves = [s, v] + list(upd.parameters())
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(3):
            out = upd(s, v)
            torch.autograd.grad(out, leaves, gs, retain_graph=True)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        if whole:
            out = upd(s, v)
        got = torch.autograd.grad(out, leaves, gs)
    for k in range(4):
        with torch.no_grad():
            for t in gs + ([s, v] if whole else []):
                t.normal_()
        torch.ones(1 << 14, dtype=torch.int64, pin_memory=True)
        g.replay()
        torch.cuda.synchronize()
        want = torch.autograd.grad(upd(s, v), leaves, gs)
        for q, (a, b) in enumerate(zip(got, want)):
            assert (a - b).norm() <= 2e-5 * b.norm() + 1e-30, (k, q)


def test_blocks_run_on_their_tensors_device(gpu, monkeypatch):
    """The blocks' kernels are launched with their tensors' device made current, as
    torch's operations are (one device here: the guard is seen to be around them);
    tensors of two devices are refused."""
    print("[case] device of the blocks", flush=True)
    model, C = pkg_mod("model"), pkg_mod("_capi")
    H, n, E = 32, 6, 20
    blk = model.PaiNNInteraction(H, 12).to(gpu)
    s, v = torch.randn(n, H, device=gpu), torch.randn(n, 3, H, device=gpu)
    inside, launches = [], []
    guard, handle = torch.cuda.device_of, C.stream_handle

    class Guard(guard):
        def __init__(self, t):
            super().__init__(t)
            self.seen = t.device

        def __enter__(self):
            inside.append(self.seen)
            return super().__enter__()

        def __exit__(self, *a):
            inside.pop()
            return super().__exit__(*a)

    def record(stream=None):
        launches.append(list(inside))
        return handle(stream)

    monkeypatch.setattr(torch.cuda, "device_of", Guard)
    monkeypatch.setattr(C, "stream_handle", record)
    with torch.no_grad():
        blk(s, v, torch.randint(0, n, (2, E), device=gpu), torch.randn(E, 12, device=gpu),
            torch.randn(E, 3, device=gpu))
    assert len(launches) == 3 and all(got == [s.device] for got in launches), launches
    monkeypatch.undo()
    blk.update.update_mlp[2].cpu()
    with pytest.raises(RuntimeError):
        blk.update(s, v)
