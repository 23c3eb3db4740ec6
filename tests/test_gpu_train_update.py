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
