"""The update block of the training pass in one launch, forward, tangent, adjoint
and the adjoint's tangent, against float64 autograd of the plain formula."""
import pytest
import torch

from conftest import pkg_mod

pytestmark = pytest.mark.gpu


def _plain(s, v, w):
    W1, b1, W2, b2, M = w
    H = s.shape[1]
    x = torch.cat([s, v.pow(2).sum(1).sqrt()], 1)
    y = torch.nn.functional.silu(x @ W1.T + b1) @ W2.T + b2
    ds, g1, g2 = y[:, :H], y[:, H:2 * H], y[:, 2 * H:]
    return s + ds, v * g1[:, None] + (M @ v) * g2[:, None]


@pytest.mark.parametrize("H", [32, 64, 128])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 50])
def test_update_block_and_its_derivatives(gpu, n, H):
    """Edges of the 16-atom tile.  1e-5 of the norm: sums of up to 384 float32
    products, whose error is about sqrt(384) 2^-24 = 1.2e-6, through two layers."""
    print(f"[case] train update n{n} H{H}", flush=True)
    train = pkg_mod("train")
    g = torch.Generator().manual_seed(n + H)
    r = lambda *sh: torch.randn(*sh, generator=g)
    w = (r(H, 2 * H) / (2 * H) ** 0.5, 0.1 * r(H), r(3 * H, H) / H ** 0.5, 0.1 * r(3 * H), r(3, 3))
    s, v, ds, dv, gs, gv, dgs, dgv = (r(n, H) if k % 2 == 0 else r(n, 3, H) for k in range(8))
    wd = tuple(t.double() for t in w)
    d = lambda *ts: tuple(t.double() for t in ts)

    def vjp(s, v, gs, gv):
        with torch.enable_grad():
            if not s.requires_grad:
                s, v = s.requires_grad_(True), v.requires_grad_(True)
            return torch.autograd.grad(_plain(s, v, wd), (s, v), (gs, gv), create_graph=True)

    out, dout = torch.autograd.functional.jvp(lambda a, b: _plain(a, b, wd), d(s, v), d(ds, dv))
    adj, dadj = torch.autograd.functional.jvp(vjp, d(s, v, gs, gv), d(ds, dv, dgs, dgv))
    dev = lambda *ts: tuple(t.to(gpu) for t in ts)
    wg = dev(*w)

    def close(a, b, what):
        assert (a.cpu().double() - b.detach()).norm() <= 1e-5 * b.detach().norm(), what

    both = train._update(wg, *dev(s, v), None, *dev(ds, dv))
    first = train._update(wg, *dev(s, v))
    then = train._update(wg, None, v.to(gpu), first, *dev(ds, dv), primal=False)
    for o in (both, {**first, **then}):
        for k, ref in (("s_out", out[0]), ("v_out", out[1]), ("ds_out", dout[0]),
                       ("dv_out", dout[1])):
            close(o[k], ref, k)
    lay = dict(both, v_m=v.to(gpu), dvm=dv.to(gpu))
    one, none = train._update_adjoint(wg, lay, *dev(gs, gv))
    two, tan = train._update_adjoint(wg, lay, *dev(gs, gv, dgs, dgv))
    assert none == [None] * 5
    for o in (one, two):
        close(o[2], adj[0], "gs")
        close(o[3], adj[1], "gv")
    close(tan[2], dadj[0], "dgs")
    close(tan[3], dadj[1], "dgv")


def test_zero_vectors_have_no_direction(gpu):
    print("[case] train update, zero vectors", flush=True)
    train = pkg_mod("train")
    H, n = 32, 5
    g = torch.Generator().manual_seed(0)
    r = lambda *sh: torch.randn(*sh, generator=g).to(gpu)
    w = (r(H, 2 * H), r(H), r(3 * H, H), r(3 * H), r(3, 3))
    z = torch.zeros(n, 3, H, device=gpu)
    o = train._update(w, r(n, H), z, None, r(n, H), r(n, 3, H))
    assert torch.equal(o["dxin"][:, H:], torch.zeros(n, H, device=gpu))
    lay = dict(o, v_m=z, dvm=r(n, 3, H))
    for t in sum(train._update_adjoint(w, lay, r(n, H), r(n, 3, H), r(n, H), r(n, 3, H)), []):
        assert torch.isfinite(t).all()


@pytest.mark.parametrize("H", [32, 64, 128])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 50])
def test_readout_and_its_derivatives(gpu, n, H):
    """As above: sums of up to 128 products through three layers."""
    print(f"[case] train readout n{n} H{H}", flush=True)
    train = pkg_mod("train")
    g = torch.Generator().manual_seed(7 * n + H)
    r = lambda *sh: torch.randn(*sh, generator=g)
    w = (r(H // 2, H) / H ** 0.5, 0.1 * r(H // 2), r(H // 4, H // 2) / (H / 2) ** 0.5,
         0.1 * r(H // 4), r(1, H // 4), r(1))
    s, ds, seed = r(n, H), r(n, H), r(3)
    batch = torch.randint(0, 3, (n,), generator=g)
    W1, b1, W2, b2, W3, b3 = (t.double() for t in w)
    silu = torch.nn.functional.silu

    def plain(x):
        return (silu(silu(x @ W1.T + b1) @ W2.T + b2) @ W3.T + b3)[:, 0]

    def vjp(x):
        with torch.enable_grad():
            if not x.requires_grad:
                x = x.requires_grad_(True)
            return torch.autograd.grad(plain(x), x, seed.double()[batch], create_graph=True)[0]

    eps = plain(s.double())
    gs, dgs = torch.autograd.functional.jvp(vjp, s.double(), ds.double())
    h4 = lambda x: silu(silu(x @ W1.T + b1) @ W2.T + b2)
    _, dh4 = torch.autograd.functional.jvp(h4, s.double(), ds.double())
    wg = tuple(t.to(gpu) for t in w)

    def close(a, b, what):
        assert (a.cpu().double() - b.detach()).norm() <= 1e-5 * b.detach().norm(), what

    both = train._readout(wg, s.to(gpu), None, ds.to(gpu))
    first = train._readout(wg, s.to(gpu))
    then = train._readout(wg, None, first, ds.to(gpu), primal=False)
    for o in (both, {**first, **then}):
        close(o["eps"], eps, "eps")
        close(o["h4"], h4(s.double()), "h4")
        close(o["dh4"], dh4, "dh4")
    sg, bg = seed.to(gpu), batch.to(gpu)
    one, none = train._readout_adjoint(wg, both, sg, bg, False)
    two, tan = train._readout_adjoint(wg, both, sg, bg, True)
    assert none == [None] * 3
    for o in (one, two):
        assert torch.equal(o[0][:, 0].cpu(), seed[batch]) and not o[0][:, 1:].any()
        close(o[3], gs, "gs")
    close(tan[2], dgs, "dgs")


@pytest.mark.parametrize("n,H", [(1, 4), (300, 20), (65, 128)])
def test_elementwise_parts_for_other_products(gpu, n, H):
    """The update block's elementwise entry points against their formulas in float64
    (1e-6 of the norm: a few roundings of each element), with a zero vector."""
    print(f"[case] update parts n{n} H{H}", flush=True)
    C = pkg_mod("_capi")
    g = torch.Generator().manual_seed(n + H)
    r = lambda *sh: torch.randn(*sh, generator=g)
    s, v, ds, dv = r(n, H), r(n, 3, H), r(n, H), r(n, 3, H)
    y, dy, gx, dgx = r(n, 3 * H), r(n, 3 * H), r(n, 2 * H), r(n, 2 * H)
    gs, gv, dgs, dgv, M = r(n, H), r(n, 3, H), r(n, H), r(n, 3, H), r(3, 3)
    v[0, :, 1] = 0.0
    D = lambda t: t.double()
    S, V, dS, dV, Y, dY, GX, dGX, GS, GV, dGS, dGV, Md = map(D, (s, v, ds, dv, y, dy, gx, dgx, gs, gv,
                                                                 dgs, dgv, M))
    part = lambda t, k: t[:, k * H:(k + 1) * H]
    up = lambda t: t[:, None]
    nrm = V.pow(2).sum(1).sqrt()
    over = torch.where(nrm > 0, 1 / nrm, torch.zeros_like(nrm))
    dn = (V * dV).sum(1) * over
    MV, dMV, g1, g2, dg1, dg2 = Md @ V, Md @ dV, part(Y, 1), part(Y, 2), part(dY, 1), part(dY, 2)
    want = {
        "xin": torch.cat([S, nrm], 1), "s": S + part(Y, 0), "v": V * up(g1) + MV * up(g2), "mv": MV,
        "dxin": torch.cat([dS, dn], 1), "ds": dS + part(dY, 0), "dmv": dMV,
        "dv": dV * up(g1) + V * up(dg1) + dMV * up(g2) + MV * up(dg2),
        "gy": torch.cat([GS, (GV * V).sum(1), (GV * MV).sum(1)], 1),
        "dgy": torch.cat([dGS, (dGV * V + GV * dV).sum(1), (dGV * MV + GV * dMV).sum(1)], 1),
        "gvg2": GV * up(g2), "dgvg2": dGV * up(g2) + GV * up(dg2),
    }
    gn, dgn, unit = part(GX, 1), part(dGX, 1), V * up(over)
    dunit = dV * up(over) - V * up(dn * over * over)
    want.update(gs=GS + part(GX, 0), dgs=dGS + part(dGX, 0),
                gv=GV * up(g1) + Md.T @ want["gvg2"] + up(gn) * unit,
                dgv=dGV * up(g1) + GV * up(dg1) + Md.T @ want["dgvg2"] + up(dgn) * unit
                + up(gn) * dunit)
    ins = {k: t.to(gpu) for k, t in dict(s=s, v=v, ds=ds, dv=dv, y=y, dy=dy, gx=gx, dgx=dgx, gs=gs,
                                         gv=gv, dgs=dgs, dgv=dgv, M=M).items()}
    out = {k: torch.full(t.shape, float("nan"), dtype=torch.float32, device=gpu)
           for k, t in want.items()}

    def call(name, *args):
        ptrs = [C.ptr(ins[a] if kind == "i" else out[a]) for kind, a in (q.split(".") for q in args)]
        C.check(name, getattr(C.lib(), "mlff_update_" + name)(C.stream_handle(), n, H, *ptrs))

    call("norm", "i.s", "i.v", "o.xin")
    call("apply", "i.M", "i.y", "i.s", "i.v", "o.s", "o.v", "o.mv")
    call("norm_tangent", "i.v", "o.xin", "i.ds", "i.dv", "o.dxin")
    call("apply_tangent", "i.M", "i.y", "i.dy", "i.ds", "i.v", "i.dv", "o.mv", "o.ds", "o.dv", "o.dmv")
    call("gate_adjoint", "i.gs", "i.gv", "i.v", "o.mv", "i.dgs", "i.dgv", "i.dv", "o.dmv", "o.gy", "o.dgy")
    call("input_adjoint", "i.M", "i.gx", "i.gs", "i.gv", "i.y", "i.v", "o.xin", "i.dgx", "i.dgs", "i.dgv",
         "i.dy", "i.dv", "o.dxin", "o.gs", "o.gv", "o.gvg2", "o.dgs", "o.dgv", "o.dgvg2")
    for k, ref in want.items():
        assert (out[k].cpu().double() - ref).norm() <= 1e-6 * ref.norm(), k
