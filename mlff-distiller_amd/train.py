"""Force-matching training on the GPU: hand-derived second-order pass.

The reference trains with torch autograd double backward
(models/distillation_wrapper.py:86-91, training/trainer.py:325-328, and the
compact recipe scripts/train_compact_models.py:229-372 with loss
wE * MSE(E) + wF * MSE(F), :340-342).  Here the gradient of the loss with
respect to the weights is formed explicitly:

  dL/dtheta = sum_b dL/dE_b dE_b/dtheta  -  d/dtheta < lambda, grad_x E >,
  lambda = dL/dF.

The first term is the reverse (adjoint) pass with parameter gradients; the
second is the tangent of that reverse pass along the position direction
lambda (forward-over-reverse).  Both come from one reverse pass seeded with
unit structure weights: its tangent gives the second term, and because
structures do not interact the first term is the same pass's parameter
terms with every atom or pair row scaled by dL/dE of its structure.

Where the work runs:
* edge- and pair-sized parts on HIP kernels (mlff_train_message,
  mlff_train_message_adjoint, mlff_train_pair_grad): the message gathers of
  the forward pass and its tangent as receiver rows in ascending neighbour
  order, the adjoint gathers the same way, and the filter-output gradients
  per unordered pair from both endpoints -- no scatter-adds, no atomics;
* per-structure energies and the embedding gradient by fixed-order segment
  sums (mlff_segment_sum);
* the update block and the readout with their products, and their reverses,
  on one kernel each (mlff_train_update, mlff_train_readout and their
  adjoints), primal and tangent together;
* weight gradients on a split-row kernel with a fixed order
  (mlff_weight_grad_partials).
Every reduction runs in a fixed order: two runs give bit-identical gradients.

The forces the loss needs come from the fused HIP evaluation of the current
weights (the trainer calls model.evaluate).  The computation is written
over unordered pairs (lo < hi), like the HIP inference kernels: a pair's
filter is evaluated once and feeds both directed edges.  float32 on the
device; energies are summed in float64.
"""

from __future__ import annotations

import ctypes
import functools
import math
import weakref
from dataclasses import dataclass
from typing import Dict, Optional, Sequence

import numpy as np
import torch

from . import _capi as C

Tensor = torch.Tensor
EPS = 1e-8   # edge_vector / (d + 1e-8), student_model.py:715


@dataclass
class PairGraph:
    """Receiver CSR of a structure-sorted batch and its unordered pairs."""
    row_ptr: Tensor          # [N+1] int32
    col: Tensor              # [E] int32, ascending within a row
    edge_pair: Tensor        # [E] int32, pair of each directed edge
    lo: Tensor               # [P] int64 (lo < hi)
    hi: Tensor               # [P] int64
    lo32: Tensor             # [P] int32
    hi32: Tensor             # [P] int32
    shift: Optional[Tensor]  # [P,3] float shift vector (already times the cell) or None
    batch: Tensor            # [N] int64 structure of each atom
    mol_ptr: Tensor          # [B+1] int32
    n_structures: int


def pair_graph_from_csr(row_ptr: Tensor, col: Tensor, batch: Tensor, n_structures: int,
                        shift_vec: Optional[Tensor] = None, n_pairs: Optional[int] = None,
                        mol_ptr: Optional[Tensor] = None) -> PairGraph:
    """Pairs (row < col) of a symmetric receiver CSR with rows in ascending
    column order, and the pair of every directed edge: an upper edge
    (row < col) numbers its pair in CSR order; a lower edge takes the
    number of its reverse edge, found by a binary search of the sorted
    (row, col) keys.  With the pair count (``n_pairs``, known on the host
    when no edge is a self-image) and the structure offsets (``mol_ptr``)
    given, nothing here waits for the device."""
    dev = col.device
    n = row_ptr.numel() - 1
    E = col.numel()
    deg = (row_ptr[1:] - row_ptr[:-1]).long()
    row = torch.repeat_interleave(torch.arange(n, device=dev), deg, output_size=E)
    colL = col.long()
    up = colL > row
    up_id = torch.cumsum(up.to(torch.int64), 0) - 1
    key = row * n + colL
    rev = torch.searchsorted(key, colL * n + row)
    edge_pair = torch.where(up, up_id, up_id[rev]).to(torch.int32)
    if n_pairs is None:
        lo, hi = row[up], colL[up]
        sv = None if shift_vec is None else shift_vec[up].contiguous()
    else:
        # every upper edge to its pair slot; the other edges to a spare slot
        dst = torch.where(up, up_id, torch.full_like(up_id, n_pairs))
        pick = lambda v: torch.empty(n_pairs + 1, dtype=v.dtype, device=dev).scatter_(
            0, dst, v)[:n_pairs]
        lo, hi = pick(row), pick(colL)
        sv = None
        if shift_vec is not None:
            sv = torch.empty(n_pairs + 1, 3, dtype=shift_vec.dtype, device=dev).index_copy_(
                0, dst, shift_vec)[:n_pairs].contiguous()
    if mol_ptr is None:
        sizes = torch.bincount(batch, minlength=n_structures)
        mol_ptr = torch.zeros(n_structures + 1, dtype=torch.int32, device=dev)
        mol_ptr[1:] = torch.cumsum(sizes, 0).to(torch.int32)
    return PairGraph(row_ptr.to(torch.int32).contiguous(), col.to(torch.int32).contiguous(),
                     edge_pair.contiguous(), lo, hi, lo.to(torch.int32).contiguous(),
                     hi.to(torch.int32).contiguous(), sv, batch.long(),
                     mol_ptr.to(torch.int32).contiguous(), n_structures)


# device layouts of non-periodic batches by (sizes, device): the training loop
# builds a pair graph per step, usually of the same batch shape
_GRAPH_LAYOUTS: "Dict[tuple, object]" = {}


def device_graph(Z: Tensor, x: Tensor, sizes: Sequence[int], rc: float, cells=None,
                 pbc=None) -> PairGraph:
    """Pair graph of a structure-sorted batch from the HIP neighbour list."""
    from . import engine
    periodic = pbc is not None and bool(np.asarray(pbc).any())
    if periodic:
        layout = engine.make_layout(sizes, x.device, cells, pbc)
    else:
        key = (tuple(int(v) for v in sizes), str(x.device))
        layout = _GRAPH_LAYOUTS.get(key)
        if layout is None:
            if len(_GRAPH_LAYOUTS) > 16:
                _GRAPH_LAYOUTS.clear()
            layout = engine.make_layout(sizes, x.device)
            _GRAPH_LAYOUTS[key] = layout
    pos32 = x.detach().to(torch.float32).contiguous()
    batch = layout.atom_mol.long()
    if not periodic:
        # isolated structures: the neighbour-list kernels number the pairs
        # (upper edges in CSR order) and link every edge to its pair
        row_ptr, col, edge_pair, lo32, hi32 = engine.neighbor_pairs(pos32, layout, rc)
        return PairGraph(row_ptr, col, edge_pair, lo32.long(), hi32.long(), lo32, hi32, None,
                         batch, layout.mol_ptr, len(sizes))
    row_ptr, col, shift = engine.neighbor_list(pos32, layout, rc, with_shifts=True)
    cell_t = torch.as_tensor(np.asarray(cells, dtype=np.float32).reshape(-1, 3, 3),
                             device=x.device)
    n = row_ptr.numel() - 1
    deg = (row_ptr[1:] - row_ptr[:-1]).long()
    row = torch.repeat_interleave(torch.arange(n, device=x.device), deg, output_size=col.numel())
    cells_e = cell_t[batch[row]]
    sh = shift.to(torch.float32)
    shift_vec = (sh[:, 0:1] * cells_e[:, 0] + sh[:, 1:2] * cells_e[:, 1] +
                 sh[:, 2:3] * cells_e[:, 2])
    # a periodic list may hold self-image edges (no upper partner): count on the device
    return pair_graph_from_csr(row_ptr, col, batch, len(sizes), shift_vec, mol_ptr=layout.mol_ptr)


# ---------------------------------------------------------------------------
# HIP launches
# ---------------------------------------------------------------------------

def _p(t: Optional[Tensor]) -> int:
    return 0 if t is None else t.data_ptr()


def _dense(t: Tensor) -> Tensor:
    """t as a contiguous, 16-byte aligned float32 device buffer."""
    if t.dtype != torch.float32 or not t.is_cuda:
        raise TypeError("the training pass runs on float32 device tensors (HIP kernels)")
    if not t.is_contiguous():
        t = t.contiguous()
    if t.data_ptr() % 16:
        t = t.clone()
    return t


def _message(g: PairGraph, H: int, s, v, W, u, ds=None, dv=None, dW=None, du=None):
    """Message outputs (s + sum s_j Ws, v + sum (v_j Wv1 + sg u Wv2)) and,
    with the tangent inputs, their tangents (mlff_train_message)."""
    s, v, W, u = _dense(s), _dense(v), _dense(W), _dense(u)
    so, vo = torch.empty_like(s), torch.empty_like(v)
    dso = dvo = None
    if ds is not None:
        ds, dv, dW, du = _dense(ds), _dense(dv), _dense(dW), _dense(du)
        dso, dvo = torch.empty_like(s), torch.empty_like(v)
    C.check("mlff_train_message", C.lib().mlff_train_message(
        C.stream_handle(), H, s.shape[0], _p(g.row_ptr), _p(g.col), _p(g.edge_pair), _p(s),
        _p(v), _p(W), _p(u), _p(ds), _p(dv), _p(dW), _p(du), _p(so), _p(vo), _p(dso), _p(dvo)))
    return so, vo, dso, dvo


def _message_adjoint(g: PairGraph, H: int, gs, gv, W, dgs=None, dgv=None, dW=None):
    """gs + sum gs_j Ws, gv + sum gv_j Wv1 and, with the tangent inputs,
    their tangents (mlff_train_message_adjoint)."""
    gs, gv, W = _dense(gs), _dense(gv), _dense(W)
    go, gvo = torch.empty_like(gs), torch.empty_like(gv)
    dgo = dgvo = None
    if dgs is not None:
        dgs, dgv, dW = _dense(dgs), _dense(dgv), _dense(dW)
        dgo, dgvo = torch.empty_like(gs), torch.empty_like(gv)
    C.check("mlff_train_message_adjoint", C.lib().mlff_train_message_adjoint(
        C.stream_handle(), H, gs.shape[0], _p(g.row_ptr), _p(g.col), _p(g.edge_pair), _p(gs),
        _p(gv), _p(W), _p(dgs), _p(dgv), _p(dW), _p(go), _p(gvo), _p(dgo), _p(dgvo)))
    return go, gvo, dgo, dgvo


def _message_adjoint_scalars(g: PairGraph, H: int, gs, W, dgs=None, dW=None):
    """gs + sum gs_j Ws and, with the tangent inputs, its tangent: _message_adjoint
    for a block whose input vectors are constants
    (mlff_train_message_adjoint_scalars)."""
    gs, W, dgs, dW = _dense(gs), _dense(W), dgs if dgs is None else _dense(dgs), \
        dW if dW is None else _dense(dW)
    go = torch.empty_like(gs)
    dgo = None if dgs is None else torch.empty_like(gs)
    C.check("mlff_train_message_adjoint_scalars", C.lib().mlff_train_message_adjoint_scalars(
        C.stream_handle(), H, gs.shape[0], _p(g.row_ptr), _p(g.col), _p(g.edge_pair), _p(gs),
        _p(W), _p(dgs), _p(dW), _p(go), _p(dgo)))
    return go, dgo


def _pair_grad(g: PairGraph, H: int, u, s, v, gs, gv, du=None, ds=None, dv=None, dgs=None,
               dgv=None):
    """dL/dW per pair from both endpoints and, with the tangents, its tangent
    (mlff_train_pair_grad)."""
    P = g.lo.numel()
    u, s, v, gs, gv = _dense(u), _dense(s), _dense(v), _dense(gs), _dense(gv)
    gW = torch.empty(P, 3 * H, dtype=torch.float32, device=s.device)
    dgW = None
    if dgs is not None:
        du, ds, dv, dgs, dgv = _dense(du), _dense(ds), _dense(dv), _dense(dgs), _dense(dgv)
        dgW = torch.empty_like(gW)
    C.check("mlff_train_pair_grad", C.lib().mlff_train_pair_grad(
        C.stream_handle(), H, P, _p(g.lo32), _p(g.hi32), _p(u), _p(du), _p(s), _p(v), _p(ds),
        _p(dv), _p(gs), _p(gv), _p(dgs), _p(dgv), _p(gW), _p(dgW)))
    return gW, dgW


def _segment_sum(seg_ptr: Tensor, src: Tensor, perm: Optional[Tensor] = None,
                 f64: bool = False) -> Tensor:
    """out[k] = sum of the rows of segment k in row order (mlff_segment_sum)."""
    src = _dense(src)
    n_seg = seg_ptr.numel() - 1
    width = src[0].numel() if src.dim() > 1 else 1
    shape = (n_seg,) + tuple(src.shape[1:])
    out = torch.empty(shape, dtype=torch.float64 if f64 else torch.float32, device=src.device)
    C.check("mlff_segment_sum", C.lib().mlff_segment_sum(
        C.stream_handle(), n_seg, width, _p(seg_ptr), _p(perm), _p(src),
        _p(out) if f64 else 0, 0 if f64 else _p(out)))
    return out


# ---------------------------------------------------------------------------
# elementwise pieces and dense products
# ---------------------------------------------------------------------------

def _update(w, s, v, lay: Optional[dict] = None, ds=None, dv=None, primal: bool = True):
    """The update block on inputs (s, v) and, with (ds, dv), its tangent, in one
    launch (mlff_train_update); ``primal`` False: the tangent of the pass stored
    in ``lay``.  w = (W1, b1, W2, b2, M), dense.  Returns what the reverse pass
    needs, outputs included (s_out, v_out, ds_out, dv_out)."""
    n, _, H = v.shape
    new = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=v.device)
    out = {}
    if primal:
        out.update(xin=new(n, 2 * H), a2=new(n, H), h2=new(n, H), y=new(n, 3 * H),
                   Mv=new(n, 3, H), s_out=new(n, H), v_out=new(n, 3, H))
    if ds is not None:
        out.update(dxin=new(n, 2 * H), da2=new(n, H), dh2=new(n, H), dy=new(n, 3 * H),
                   dMv=new(n, 3, H), ds_out=new(n, H), dv_out=new(n, 3, H))
    src = out if primal else lay
    P = C.ptr
    W1, b1, W2, b2, M = w
    C.check("mlff_train_update", C.lib().mlff_train_update(
        C.stream_handle(), int(primal) + 2 * (ds is not None), n, H, P(s), P(v), P(ds), P(dv),
        P(W1), P(b1), P(W2), P(b2), P(M), P(src["xin"]), P(src["a2"]), P(src["h2"]), P(src["y"]),
        P(src["Mv"]), P(out.get("s_out")), P(out.get("v_out")), P(out.get("dxin")),
        P(out.get("da2")), P(out.get("dh2")), P(out.get("dy")), P(out.get("dMv")),
        P(out.get("ds_out")), P(out.get("dv_out"))))
    return out


def _update_adjoint(w, lay: dict, gs, gv, dgs=None, dgv=None):
    """Adjoint of _update from the output gradients and, with (dgs, dgv), its
    tangent (mlff_train_update_adjoint): ([gy, ga, gs_m, gv_m, gvg2], the same of
    the tangent or Nones)."""
    n, _, H = gv.shape
    new = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=gv.device)
    outs = lambda: [new(n, 3 * H), new(n, H), new(n, H), new(n, 3, H), new(n, 3, H)]
    T = dgs is not None
    out, dout = outs(), outs() if T else [None] * 5
    t = (lambda k: lay[k]) if T else (lambda k: None)
    W1, _, W2, _, M = w
    C.check("mlff_train_update_adjoint", C.lib().mlff_train_update_adjoint(
        C.stream_handle(), n, H, *[C.ptr(q) for q in (
            gs, gv, dgs, dgv, lay["v_m"], lay["Mv"], lay["y"], lay["a2"], lay["xin"], t("dvm"),
            t("dMv"), t("dy"), t("da2"), t("dxin"), W1, W2, M, *out, *dout)]))
    return out, dout


def _fit(t: Tensor, shape: tuple) -> Tensor:
    """t as a dense buffer of the shape that the kernels assume: a layer with fewer
    hidden channels is filled up with zeros, as in the weight blob.  A zero channel
    has silu(0) = 0 and zero weights behind it, so it changes no other value."""
    if t.shape != shape:
        if t.dim() != len(shape) or any(a > b for a, b in zip(t.shape, shape)):
            raise ValueError(f"layer of shape {tuple(t.shape)} in place of {shape}")
        pad = [q for a, b in zip(reversed(t.shape), reversed(shape)) for q in (0, b - a)]
        t = torch.nn.functional.pad(t, pad)
    return _dense(t)


@functools.lru_cache(maxsize=None)
def _update_shapes(H: int):
    return ((".update_mlp.0.weight", (H, 2 * H)), (".update_mlp.0.bias", (H,)),
            (".update_mlp.2.weight", (3 * H, H)), (".update_mlp.2.bias", (3 * H,)),
            (".mixing_matrix", (3, 3)))


@functools.lru_cache(maxsize=None)
def _readout_shapes(H: int):
    return (("energy_head.0.weight", (H // 2, H)), ("energy_head.0.bias", (H // 2,)),
            ("energy_head.2.weight", (H // 4, H // 2)), ("energy_head.2.bias", (H // 4,)),
            ("energy_head.4.weight", (1, H // 4)), ("energy_head.4.bias", (1,)))


def _update_weights(p: Dict[str, Tensor], upre: str):
    H = p["embedding.weight"].shape[1]
    return tuple([_fit(p[upre + k], shape) for k, shape in _update_shapes(H)])


def _readout_weights(p: Dict[str, Tensor]):
    H = p["embedding.weight"].shape[1]
    return tuple([_fit(p[k], shape) for k, shape in _readout_shapes(H)])


def _readout(w, s, c: Optional[dict] = None, ds=None, primal: bool = True):
    """The readout of s and, with ds, its tangent, in one launch
    (mlff_train_readout); w = (W1, b1, W2, b2, W3, b3), dense.  ``primal`` False:
    the tangent of the pass stored in ``c``."""
    n, H = (s if primal else ds).shape
    dev = w[0].device
    new = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=dev)
    out = {}
    if primal:
        out.update(r1=new(n, H // 2), h3=new(n, H // 2), r2=new(n, H // 4), h4=new(n, H // 4),
                   eps=new(n))
    if ds is not None:
        out.update(dr1=new(n, H // 2), dh3=new(n, H // 2), dr2=new(n, H // 4),
                   dh4=new(n, H // 4))
    src = out if primal else c
    keys = ("dr1", "dh3", "dr2", "dh4")
    C.check("mlff_train_readout", C.lib().mlff_train_readout(
        C.stream_handle(), int(primal) + 2 * (ds is not None), n, H, C.ptr(s), C.ptr(ds),
        *[C.ptr(t) for t in w], C.ptr(src["r1"]), C.ptr(src["h3"]), C.ptr(src["r2"]),
        C.ptr(src["h4"]), C.ptr(src.get("eps")), *[C.ptr(out.get(k)) for k in keys]))
    return out


def _readout_adjoint(w, c: dict, seed, batch, T: bool):
    """(g4, gr2, gr1, gs) from the structures' seeds and, with T, the tangents
    (dgr2, dgr1, dgs) or Nones (mlff_train_readout_adjoint)."""
    r1, r2 = c["r1"], c["r2"]
    n, H = r1.shape[0], 2 * r1.shape[1]
    new = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=r1.device)
    outs = lambda: [new(n, H // 4), new(n, H // 2), new(n, H)]
    g4, out, dout = new(n, 4), outs(), outs() if T else [None] * 3
    C.check("mlff_train_readout_adjoint", C.lib().mlff_train_readout_adjoint(
        C.stream_handle(), n, H, C.ptr(seed), C.ptr(batch), C.ptr(r1), C.ptr(r2),
        C.ptr(c["dr1"] if T else None), C.ptr(c["dr2"] if T else None), C.ptr(w[0]), C.ptr(w[2]),
        C.ptr(w[4]), C.ptr(g4), *[C.ptr(t) for t in out + dout]))
    return (g4, *out), dout


def _silu_call(a, da=None, g=None, dg=None, h=False, dh=False, dga=False):
    a = _dense(a)
    opt = lambda t: None if t is None else _dense(t)
    da, g, dg = opt(da), opt(g), opt(dg)
    outs = [torch.empty_like(a) if want else None for want in (h, dh, dga)]
    C.check("mlff_silu_chain", C.lib().mlff_silu_chain(
        C.stream_handle(), a.numel(), C.ptr(a), C.ptr(da), C.ptr(g), C.ptr(dg),
        C.ptr(outs[0]), C.ptr(outs[1]), None, C.ptr(outs[2])))
    return [o for o in outs if o is not None][0]


def _silu(x):
    """silu(x) = x sigmoid(x) (mlff_silu_chain)."""
    return _silu_call(x, h=True)


def _silu_d(x, t):
    """silu'(x) t: a tangent along t, or the adjoint of a gradient t."""
    return _silu_call(x, da=t, dh=True)


def _silu_dd(x, g, dx, dg=None):
    """dg silu'(x) + g silu''(x) dx: the tangent of the adjoint g silu'(x)
    along (dx, dg); dg None is zero."""
    return _silu_call(x, da=dx, g=g, dg=dg, dga=True)


# prepared filter weights per (W1, W2) tensor pair: W1 padded to 16 or 32
# columns, W2 and its transpose as three bf16 planes each, and the transpose
# itself.  An entry belongs to
# the two tensor objects themselves (weak references: a tensor allocated later at
# a freed one's address, or under its id, never matches) and is remade when the
# optimizer has written either tensor (its version counter moved).
_FILTER_W: Dict[tuple, tuple] = {}


def _filter_weights(p: Dict[str, Tensor], pre: str):
    W1o, W2o = p[pre + ".0.weight"], p[pre + ".2.weight"]
    key = (id(W1o), id(W2o))
    state = (W1o.data_ptr(), W2o.data_ptr(), W1o._version, W2o._version)
    ent = _FILTER_W.get(key)
    same = ent is not None and ent[0]() is W1o and ent[1]() is W2o
    if same and ent[2] == state:
        return ent[3:]
    W1, W2 = _dense(W1o), _dense(W2o)
    H, R = W1.shape
    if W2.shape != (3 * H, H):
        raise RuntimeError("filter layers do not match: W2 must be [3H, H]")
    RP = 16 if R <= 16 else 32
    if len(_FILTER_W) > 64:
        for k in [k for k, e in _FILTER_W.items() if e[0]() is None or e[1]() is None]:
            del _FILTER_W[k]
    if same and ent[3].shape == (H, RP):
        # the same tensors, written by the optimizer: refill the buffers in place
        w1p, planes, planes_t, w2t = ent[3:]
    else:
        w1p = torch.empty(H, RP, dtype=torch.float32, device=W1.device)
        planes = torch.empty(3 * W2.numel(), dtype=torch.int16, device=W2.device)
        planes_t = torch.empty_like(planes)
        w2t = torch.empty(H, 3 * H, dtype=torch.float32, device=W2.device)
    C.check("mlff_filter_planes", C.lib().mlff_filter_planes(
        C.stream_handle(), H, R, C.ptr(W1), C.ptr(W2), C.ptr(w1p), C.ptr(planes),
        C.ptr(planes_t), C.ptr(w2t)))
    _FILTER_W[key] = (weakref.ref(W1o), weakref.ref(W2o), state, w1p, planes, planes_t, w2t)
    return w1p, planes, planes_t, w2t


def _filter(p: Dict[str, Tensor], pre: str, x: Tensor, a: Optional[Tensor] = None):
    """The filter MLP on the fused pair kernel (mlff_train_filter).  Forward
    (a None): x = e gives (a1, h, W) with a1 = e W1^T + b1, h = silu(a1),
    W = h W2^T + b2.  Tangent: x = de and a = a1 give (da1, dh, dW) with
    da1 = de W1^T, dh = silu'(a1) da1, dW = dh W2^T."""
    w1p, planes, _, _ = _filter_weights(p, pre)
    x = _dense(x)
    P, R = x.shape
    H = p[pre + ".0.weight"].shape[0]
    if w1p.shape[0] != H or planes.numel() != 3 * p[pre + ".2.weight"].numel():
        raise RuntimeError("prepared filter weights do not match the layer")
    a_out = torch.empty(P, H, dtype=torch.float32, device=x.device)
    h_out = torch.empty_like(a_out)
    w_out = torch.empty(P, 3 * H, dtype=torch.float32, device=x.device)
    tan = a is not None
    b1 = None if tan else _dense(p[pre + ".0.bias"])
    b2 = None if tan else _dense(p[pre + ".2.bias"])
    a = _dense(a) if tan else None
    C.check("mlff_train_filter", C.lib().mlff_train_filter(
        C.stream_handle(), int(tan), H, P, R, C.ptr(x), C.ptr(w1p), C.ptr(b1), C.ptr(planes),
        C.ptr(b2), C.ptr(a), C.ptr(a_out), C.ptr(h_out), C.ptr(w_out)))
    return a_out, h_out, w_out


def _filters(p: Dict[str, Tensor], L: int, e: Tensor, de: Optional[Tensor] = None):
    """The filter MLPs of all L blocks on the basis e and, with de, their
    tangents, in one launch (mlff_train_filters): a list of (a1, h, W) or
    (a1, h, W, da1, dh, dW) per block, as _filter gives them."""
    e = _dense(e)
    de = None if de is None else _dense(de)
    P, R = e.shape
    H = p["interactions.0.message.rbf_to_scalar.0.weight"].shape[0]
    got, rows, keep = [], [], []
    for k in range(L):
        pre = f"interactions.{k}.message.rbf_to_scalar"
        w1p, planes, _, _ = _filter_weights(p, pre)
        if w1p.shape[0] != H or planes.numel() != 3 * p[pre + ".2.weight"].numel():
            raise RuntimeError("prepared filter weights do not match the layer")
        b1, b2 = _dense(p[pre + ".0.bias"]), _dense(p[pre + ".2.bias"])
        out = [torch.empty(P, c, dtype=torch.float32, device=e.device)
               for c in (H, H, 3 * H) * (1 if de is None else 2)]
        got.append(out)
        keep += [w1p, planes, b1, b2]
        rows += [C.ptr(t) for t in (w1p, b1, planes, b2, *out)] + [0] * (6 - len(out))
    for at in range(0, L, 8):   # at most 8 blocks per launch
        n = min(8, L - at)
        table = (ctypes.c_void_p * (10 * n))(*rows[10 * at:10 * (at + n)])
        C.check("mlff_train_filters", C.lib().mlff_train_filters(
            C.stream_handle(), H, n, P, R, C.ptr(e), C.ptr(de), table))
    return got


def _filter_adjoint(p: Dict[str, Tensor], pre: str, gW: Tensor, a1: Tensor,
                    dgW: Optional[Tensor] = None, da1: Optional[Tensor] = None):
    """Reverse of the filter's first layer on the fused pair kernel
    (mlff_train_filter_adjoint): ga1 = silu'(a1) (gW W2) and, with the
    tangent (dgW, da1), dga1 = silu'(a1) (dgW W2) + silu''(a1) da1 (gW W2).
    Returns (ga1, dga1 or None)."""
    _, _, planes_t, w2t = _filter_weights(p, pre)
    gW, a1 = _dense(gW), _dense(a1)
    P, H = a1.shape
    if w2t.shape != (H, 3 * H) or gW.shape != (P, 3 * H):
        raise RuntimeError("filter adjoint operands do not match the layer")
    tan = dgW is not None
    ga = torch.empty(P, H, dtype=torch.float32, device=a1.device)
    dga = torch.empty_like(ga) if tan else None
    dgW, da1 = (_dense(dgW), _dense(da1)) if tan else (None, None)
    if H > 32:
        C.check("mlff_train_filter_adjoint_x6", C.lib().mlff_train_filter_adjoint_x6(
            C.stream_handle(), H, P, C.ptr(gW), C.ptr(dgW), C.ptr(planes_t), C.ptr(a1),
            C.ptr(da1), C.ptr(ga), C.ptr(dga)))
        return ga, dga
    C.check("mlff_train_filter_adjoint", C.lib().mlff_train_filter_adjoint(
        C.stream_handle(), int(tan), H, P, C.ptr(gW), C.ptr(dgW), C.ptr(w2t), C.ptr(a1),
        C.ptr(da1), C.ptr(ga), C.ptr(dga)))
    return ga, dga


def _edge_features(d, centers, widths, rc):
    """e_k(d) = exp(-(d-mu_k)^2 / w_k^2) * 0.5 (cos(pi d/rc) + 1) [d < rc]
    (student_model.py:249-253, 285-290, 720-722) and de/dd."""
    diff = d.unsqueeze(-1) - centers
    gamma = 1.0 / widths ** 2
    phi = torch.exp(-gamma * diff ** 2)
    inside = (d < rc).to(d.dtype).unsqueeze(-1)
    arg = math.pi * d.unsqueeze(-1) / rc
    fc = 0.5 * (torch.cos(arg) + 1.0) * inside
    dfc = -0.5 * (math.pi / rc) * torch.sin(arg) * inside
    return phi * fc, (-2.0 * gamma * diff * phi) * fc + phi * dfc


def _geometry(g: PairGraph, x: Tensor, centers: Tensor, widths: Tensor, rc: float,
              lam: Optional[Tensor] = None):
    """Pair geometry and basis on one HIP launch (mlff_train_geometry):
    (vec, d, den, u, e, de) with vec = x[hi] - x[lo] (+ shift), d = |vec|,
    den = d + EPS, u = vec / den, e = _edge_features(d) and de = de/dd; with
    a position direction ``lam``, the tangent (dd, du, de_t) instead."""
    P = g.lo32.numel()
    R = centers.numel()
    dev = x.device
    f = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=dev)
    shift = None if g.shift is None else _dense(g.shift.to(torch.float32))
    x, centers, widths = _dense(x), _dense(centers), _dense(widths)
    lam = None if lam is None else _dense(lam)
    if lam is None:
        outs = (f(P, 3), f(P), f(P), f(P, 3), f(P, R), f(P, R))
        ptrs = [C.ptr(t) for t in outs] + [None] * 3
    else:
        outs = (f(P), f(P, 3), f(P, R))
        ptrs = [None] * 6 + [C.ptr(t) for t in outs]
    C.check("mlff_train_geometry", C.lib().mlff_train_geometry(
        C.stream_handle(), P, R, C.ptr(x), C.ptr(lam), C.ptr(g.lo32), C.ptr(g.hi32),
        C.ptr(shift), C.ptr(centers), C.ptr(widths), float(rc), EPS, *ptrs))
    return outs


def _edge_feature_param_derivs(d, centers, widths, rc):
    """de_k/dmu_k, de_k/dw_k and their d-derivatives, each [P, R]
    (learnable_rbf, student_model.py:226-236): with phi = exp(-(d-mu)^2/w^2),
    dphi/dmu = 2 gamma (d-mu) phi and dphi/dw = 2 (d-mu)^2 phi / w^3."""
    diff = d.unsqueeze(-1) - centers
    gamma = 1.0 / widths ** 2
    phi = torch.exp(-gamma * diff ** 2)
    inside = (d < rc).to(d.dtype).unsqueeze(-1)
    arg = math.pi * d.unsqueeze(-1) / rc
    fc = 0.5 * (torch.cos(arg) + 1.0) * inside
    dfc = -0.5 * (math.pi / rc) * torch.sin(arg) * inside
    w3 = widths ** 3
    A = 2.0 * gamma * diff * phi
    Bw = 2.0 * diff ** 2 * phi / w3
    dA = 2.0 * gamma * phi * (1.0 - 2.0 * gamma * diff ** 2)
    dBw = (2.0 * diff * phi / w3) * (2.0 - 2.0 * gamma * diff ** 2)
    return fc * A, fc * Bw, dfc * A + fc * dA, dfc * Bw + fc * dBw


def _wg_operand(t: Tensor) -> Tensor:
    """A [K, C] float32 operand of mlff_weight_grad: unit column stride, row
    stride and C multiples of 4 (zero columns appended), 16-byte aligned."""
    t = t.reshape(t.shape[0], math.prod(t.shape[1:]))
    if t.shape[1] % 4:
        t = torch.nn.functional.pad(t, (0, 4 - t.shape[1] % 4))
    if t.stride(1) != 1 or t.stride(0) % 4:
        t = t.contiguous()
    if t.data_ptr() % 16:
        t = t.clone()
    return t


_WG_WS: Dict[tuple, int] = {}   # workspace floats of mlff_weight_grad by (K, M, N)
_WG_S: Dict[tuple, int] = {}    # partial sums of mlff_weight_grad by (K, M, N)


class _WgGroup:
    """Weight gradients that are finished later: the partial sums of all are
    added in one launch (mlff_weight_grad_reduce_group), and those of the short
    ones (the atoms' rows) are formed in one launch per kind
    (mlff_weight_grad_group).  The outputs _wgrad returns with a group hold
    their values only after flush(); operands and partials are kept until then."""

    def __init__(self):
        self.rows = []
        self.keep = []
        self.short = {}     # kind: [(K, M, N, operands, out, bias)]

    def add(self, S: int, n4: int, part: int, out: int, buf: Tensor):
        self.rows.append((S, n4, part, out))
        self.keep.append(buf)

    def flush(self):
        words, launches = [], []
        for kind, probs in self.short.items():
            splits = [_wg_split(*q[:3]) for q in probs]
            part = torch.empty(sum(S * (M * N + M) for (_, S), (_, M, N, *_) in
                                   zip(splits, probs)), dtype=torch.float32,
                               device=probs[0][3][0].device)
            self.keep.append((part, probs))
            at, first, start = part.data_ptr(), 0, len(words) // 14
            for (RW, S), (K, M, N, ops, out) in zip(splits, probs):
                a0, b0, a1, b1, w = ops
                tm, tn = (M + 63) // 64, (N + 63) // 64
                ld = lambda t: 0 if t is None else t.stride(0)
                pair = lambda x, y: x | y << 32
                words += [first, pair(K, M), pair(N, RW), pair(tm, tn), pair(S, ld(a0)),
                          pair(ld(b0), ld(a1)), ld(b1), _p(a0), _p(b0), _p(a1), _p(b1), _p(w), at,
                          at + 4 * S * M * N]
                self.rows += [(S, M * N // 4, at, out.data_ptr()),
                              (S, M // 4, at + 4 * S * M * N, out.data_ptr() + 4 * M * N)]
                at += 4 * S * (M * N + M)
                first += tm * tn * S
            launches.append((kind, len(probs), start, first))
        self.short = {}
        if not self.rows:
            return
        lib = C.lib()
        keep = self.keep[0]
        dev = (keep[0] if isinstance(keep, tuple) else keep).device
        n = len(words)
        for row in self.rows:
            words += row
        table = torch.tensor(words, dtype=torch.int64, pin_memory=True).to(dev, non_blocking=True)
        at = table.data_ptr()
        for kind, n_probs, start, blocks in launches:
            C.check("mlff_weight_grad_group", lib.mlff_weight_grad_group(
                C.stream_handle(), kind, n_probs, at + 112 * start, blocks))
        for i in range(0, len(self.rows), 256):   # at most 256 rows per launch
            rows = self.rows[i:i + 256]
            n_blocks = sum((n4 + 31) // 32 for _, n4, _, _ in rows)
            C.check("mlff_weight_grad_reduce_group", lib.mlff_weight_grad_reduce_group(
                C.stream_handle(), len(rows), at + 8 * n + 32 * i, min(n_blocks, 1 << 16)))
        self.rows, self.keep = [], []


_WG_SPLIT: Dict[tuple, tuple] = {}   # (rows per wave, partials) by (K, M, N)


def _wg_split(K: int, M: int, N: int):
    got = _WG_SPLIT.get((K, M, N))
    if got is None:
        rw, S = ctypes.c_int(), ctypes.c_int()
        C.check("mlff_weight_grad_split", C.lib().mlff_weight_grad_split(
            K, M, N, ctypes.byref(rw), ctypes.byref(S)))
        if len(_WG_SPLIT) > 4096:
            _WG_SPLIT.clear()
        got = _WG_SPLIT[(K, M, N)] = (rw.value, S.value)
    return got


def _wgrad(a0: Tensor, b0: Tensor, a1: Optional[Tensor] = None, b1: Optional[Tensor] = None,
           w: Optional[Tensor] = None, bias: bool = False, group: Optional[_WgGroup] = None,
           diff: bool = False, short: bool = False):
    """sum_k w_k (a0[k] (x) b0[k] + a1[k] (x) b1[k]) [M, N] and, with
    ``bias``, sum_k w_k a0[k] [M] over the K rows (pairs or atoms): a Linear
    layer's weight and bias gradients, on the MFMA kernel with a fixed split
    and order of the row sum (mlff_weight_grad).  Returns (weight, bias or
    None).  With ``group`` only the partial sums are launched here; the
    outputs are filled, with the same bits, by group.flush().  ``diff`` (with a
    group): (w a1 - a0) (x) b0 - a1 (x) b1 and the sum of w a1 - a0
    (mlff_weight_grad_diff_partials).  ``short`` (with a group and bias): one of
    the launch of short ones at the flush."""
    M, N = a0.shape[1], b0.shape[1]
    K = a0.shape[0]
    A0, B0 = _wg_operand(a0), _wg_operand(b0)
    A1 = B1 = None
    if a1 is not None:
        A1, B1 = _wg_operand(a1), _wg_operand(b1)
    M4, N4 = A0.shape[1], B0.shape[1]
    if short:
        wv = None if w is None else _dense(w.to(torch.float32))
        buf = torch.empty(M4 * N4 + M4, dtype=torch.float32, device=a0.device)
        if not diff and A1 is not None and wv is not None:
            raise ValueError("short weight gradients: two terms take no row weights")
        kind = 3 if diff else 2 if A1 is not None else int(wv is not None)
        group.short.setdefault(kind, []).append((K, M4, N4, (A0, B0, A1, B1, wv), buf))
        return buf[:M4 * N4].view(M4, N4)[:M, :N], buf[M4 * N4:][:M]
    lib = C.lib()
    key = (K, M4, N4)
    ws_floats = _WG_WS.get(key)
    if ws_floats is None:
        ws_floats = (int(lib.mlff_weight_grad_workspace_bytes(K, M4, N4)) + 15) // 16 * 4
        _WG_WS[key] = ws_floats
    # one allocation: workspace, then the weight gradient, then the bias
    buf = torch.empty(ws_floats + M4 * N4 + M4, dtype=torch.float32, device=a0.device)
    out = buf[ws_floats:ws_floats + M4 * N4].view(M4, N4)
    bout = buf[ws_floats + M4 * N4:] if bias else None
    wv = None
    if w is not None:
        wv = w if (w.dtype == torch.float32 and w.is_contiguous()) else w.to(torch.float32).contiguous()
    operands = (C.stream_handle(), K, M4, N4, A0.data_ptr(), A0.stride(0), B0.data_ptr(),
                B0.stride(0), C.ptr(A1), A1.stride(0) if A1 is not None else 0,
                C.ptr(B1), B1.stride(0) if B1 is not None else 0, C.ptr(wv))
    if group is None:
        C.check("mlff_weight_grad", lib.mlff_weight_grad(
            *operands, buf.data_ptr(), ws_floats * 4, out.data_ptr(), C.ptr(bout)))
    else:
        fn = "mlff_weight_grad_diff_partials" if diff else "mlff_weight_grad_partials"
        C.check(fn, getattr(lib, fn)(*operands, int(bias), buf.data_ptr(), ws_floats * 4))
        S = _WG_S.get(key)
        if S is None:
            S = _WG_S[key] = int(lib.mlff_weight_grad_partial_count(K, M4, N4))
        group.add(S, M4 * N4 // 4, buf.data_ptr(), out.data_ptr(), buf)
        if bout is not None:
            group.add(S, M4 // 4, buf.data_ptr() + S * M4 * N4 * 4, bout.data_ptr(), buf)
    if M4 != M or N4 != N:
        out = out[:M, :N]
    if bout is not None and M4 != M:
        bout = bout[:M]
    return out, bout


def _xyz_outer(a, b, a1=None, b1=None, w=None, group: Optional[_WgGroup] = None,
               diff: bool = False):
    """sum_n w_n sum_h (a[n,x,h] b[n,z,h] + a1[n,x,h] b1[n,z,h]) -> [3,3]
    (gradient of a 3x3 mixing matrix), on one partial-sum kernel
    (mlff_xyz_outer_partials) whose partials the weight-gradient reduce adds:
    at ``group``'s flush when one is given, else at once.  ``diff`` as in
    _wgrad."""
    n, _, H = a.shape
    lib = C.lib()
    S = int(lib.mlff_xyz_outer_partial_count(n))
    buf = torch.empty(12 * S + 12, dtype=torch.float32, device=a.device)
    opt = lambda t: None if t is None else _dense(t)
    a, b, a1, b1 = _dense(a), _dense(b), opt(a1), opt(b1)
    wv = None if w is None else _dense(w.to(torch.float32))
    fn = "mlff_xyz_outer_diff_partials" if diff else "mlff_xyz_outer_partials"
    C.check(fn, getattr(lib, fn)(
        C.stream_handle(), n, H, C.ptr(a), C.ptr(b), C.ptr(a1), C.ptr(b1), C.ptr(wv),
        buf.data_ptr()))
    out = buf[12 * S:]
    grp = group if group is not None else _WgGroup()
    grp.add(S, 3, buf.data_ptr(), out.data_ptr(), buf)
    if group is None:
        grp.flush()
    return out[:9].view(3, 3)


# ---------------------------------------------------------------------------
# forward (with saved activations) and its tangent
# ---------------------------------------------------------------------------

def forward(p: Dict[str, Tensor], Z: Tensor, x: Tensor, g: PairGraph, rc: float,
            lam: Optional[Tensor] = None):
    """Primal pass (student_model.py:634-757); returns (E [B] float64, cache).
    With ``lam`` [N,3] the tangent along lam is computed too, block by block
    beside the primal pass: the message kernel's tangent form gives both, so
    a block's filters are read once."""
    H = p["embedding.weight"].shape[1]
    L = len({int(k.split(".")[1]) for k in p if k.startswith("interactions.")})
    n = Z.shape[0]
    x = _dense(x.to(torch.float32))
    vec, d, den, u, e, de = _geometry(g, x, p["rbf.centers"], p["rbf.widths"], rc)
    s = p["embedding.weight"][Z].contiguous()
    v = torch.zeros(n, 3, H, dtype=torch.float32, device=x.device)
    layers = []
    cache = dict(H=H, L=L, n=n, x=x, vec=vec, d=d, den=den, u=u, e=e, de=de, layers=layers,
                 Z=Z, rc=rc, lam=None)
    t = None if lam is None else _Tangent(p, cache, lam, g, filters=True)
    filters = _filters(p, L, e, None if t is None else t.geometry[2])
    for k in range(L):
        lay = dict(zip(("a1", "h", "W", "da1", "dh", "dW"), filters[k]), s=s, v=v)
        layers.append(lay)
        if t is None:
            s_m, v_m, _, _ = _message(g, H, s, v, lay["W"], u)
        else:
            s_m, v_m = t.message(k, g)
        # PaiNNUpdate.forward (student_model.py:430-470)
        lay.update(s_m=s_m, v_m=v_m, w=_update_weights(p, f"interactions.{k}.update"))
        if t is None:
            lay.update(_update(lay["w"], s_m, v_m))
        else:
            lay.update(_update(lay["w"], s_m, v_m, None, *t.moved(k)))
            t.updated(k)
        s, v = lay["s_out"], lay["v_out"]
    cache.update(sL=s, wr=_readout_weights(p))
    if t is None:
        cache.update(_readout(cache["wr"], s))
    else:
        cache.update(_readout(cache["wr"], s, None, t.ds))
        t.finish()
    E = _segment_sum(g.mol_ptr, cache["eps"], f64=True)
    return E, cache


class _Tangent:
    """Tangent of the forward pass along the position direction lam [N,3], block
    by block behind the primal pass of each; stored in the cache."""

    def __init__(self, p: Dict[str, Tensor], c: dict, lam: Tensor, g: PairGraph,
                 filters: bool = False):
        self.p, self.c, self.lam, self.filters = p, c, lam, filters
        self.geometry = _geometry(g, c["x"], p["rbf.centers"], p["rbf.widths"], c["rc"],
                                  lam.to(torch.float32))
        f = lambda *shape: torch.zeros(*shape, dtype=torch.float32, device=c["x"].device)
        self.ds, self.dv = f(c["n"], c["H"]), f(c["n"], 3, c["H"])

    def message(self, k: int, g: PairGraph):
        """Block k's message outputs (and its filters' tangent, unless ``filters``:
        formed with the primal ones); returns the primal outputs."""
        p, c, H = self.p, self.c, self.c["H"]
        _, du, de_t = self.geometry
        lay = c["layers"][k]
        lay["ds"], lay["dv"] = self.ds, self.dv
        if not self.filters:
            lay["da1"], lay["dh"], lay["dW"] = _filter(
                p, f"interactions.{k}.message.rbf_to_scalar", de_t, lay["a1"])
        s_m, v_m, self.dsm, self.dvm = _message(g, H, lay["s"], lay["v"], lay["W"], c["u"],
                                                self.ds, self.dv, lay["dW"], du)
        return s_m, v_m

    def moved(self, k: int):
        """Tangents of block k's message outputs."""
        return self.dsm, self.dvm

    def updated(self, k: int):
        lay = self.c["layers"][k]
        lay.update(dsm=self.dsm, dvm=self.dvm)
        self.ds, self.dv = lay["ds_out"], lay["dv_out"]

    def finish(self):
        c = self.c
        dd, du, de_t = self.geometry
        c.update(lam=self.lam, dd=dd, du=du, de_t=de_t, dsL=self.ds)


def tangent(p: Dict[str, Tensor], c: dict, g: PairGraph, lam: Tensor):
    """Tangent of a finished forward pass along lam [N,3], stored in the cache."""
    t = _Tangent(p, c, lam, g)
    for k in range(c["L"]):
        t.message(k, g)
        lay = c["layers"][k]
        lay.update(_update(lay["w"], None, lay["v_m"], lay, *t.moved(k), primal=False))
        t.updated(k)
    c.update(_readout(c["wr"], None, c, t.ds, primal=False))
    t.finish()


# ---------------------------------------------------------------------------
# reverse pass (parameter gradients), optionally with its tangent
# ---------------------------------------------------------------------------

# element segments of the last element tensor seen: a training loop over one
# batch passes the same tensor every step (weak reference: a tensor made later
# at the same address never matches; the version counter catches writes)
_Z_SEG: Dict[str, tuple] = {}


def _z_segments(Z: Tensor, n_rows: int):
    """Atoms ordered by element (stable sort) and the element segments, for
    the fixed-order embedding-gradient sum."""
    ent = _Z_SEG.get("last")
    if ent is not None and ent[0]() is Z and ent[1] == (Z._version, n_rows):
        return ent[2], ent[3]
    zs, order = torch.sort(Z, stable=True)
    # first position of each element in the sorted list (no host sync)
    ptr = torch.searchsorted(zs, torch.arange(n_rows + 1, dtype=zs.dtype, device=Z.device))
    ptr, order = ptr.to(torch.int32), order.to(torch.int32)
    _Z_SEG["last"] = (weakref.ref(Z), (Z._version, n_rows), ptr, order)
    return ptr, order


def reverse(p: Dict[str, Tensor], c: dict, g: PairGraph, gE: Tensor,
            lam: Optional[Tensor] = None, gw: Optional[Tensor] = None,
            rbf_grads: bool = False, primal: bool = True, diff: bool = False):
    """Parameter gradients of sum_b gw_b E_b (gw defaults to gE) and -- with
    the tangent along ``lam`` [N,3] (reused from the cache when forward()
    already computed it for the same lam) -- the parameter gradients of
    < lam, grad_x (sum_b gE_b E_b) >.  Returns (grads, tgrads or None); without
    ``primal`` the tangent's only ({}, tgrads), with ``diff`` (lam and gw
    given) their difference (grads - tgrads, None) from two products per
    weight instead of three.

    gw is applied as a per-row weight on the gE adjoint (structures do not
    interact), so gE must then be all ones.  ``rbf_grads`` adds the basis
    centres and widths (learnable_rbf)."""
    H, L, n = c["H"], c["L"], c["n"]
    T = lam is not None
    if T and c.get("lam") is not lam:
        tangent(p, c, g, lam)
    grads: Dict[str, Tensor] = {}
    tg: Dict[str, Tensor] = {}
    dev = c["d"].device

    # the weight gradients' partial sums are added by one launch at the end
    grp = _WgGroup()

    def acc(store, name, val):
        if name in store:
            grp.flush()   # both terms must hold their values
            store[name] = store[name] + val
        else:
            store[name] = val

    def linear(name, ga, b, dga, db, w, short=True):
        """Weight and bias gradients of a Linear with adjoint ga and input b."""
        def put(store, *a, **kw):
            gw_, gb_ = _wgrad(*a, bias=True, group=grp, short=short, **kw)
            m, k = p[name + ".weight"].shape
            if gw_.shape != (m, k):   # channels that the layer has not (_fit, the seeds)
                gw_, gb_ = gw_[:m, :k], gb_[:m]
            acc(store, name + ".weight", gw_)
            acc(store, name + ".bias", gb_)

        if diff:
            put(grads, dga, b, ga, db, w=w, diff=True)
            return
        if primal:
            put(grads, ga, b, w=w)
        if T:
            put(tg, dga, b, ga, db)

    def direct(name, val, dval):
        """A gradient and its tangent's, each given as a function."""
        if diff:
            acc(grads, name, val() - dval())
            return
        if primal:
            acc(grads, name, val())
        if T:
            acc(tg, name, dval())

    gE = gE.to(torch.float32)
    w_atom = w_pair = None
    if gw is not None:
        gw = gw.to(torch.float32)
        w_atom = gw[g.batch]
        w_pair = w_atom[g.lo]
        wa = lambda t: t * w_atom.view(-1, *([1] * (t.dim() - 1)))
        wp = lambda t: t * w_pair.view(-1, *([1] * (t.dim() - 1)))
    else:
        wa = wp = lambda t: t

    # ---- readout reverse ------------------------------------------------------
    (g4, gr2, gr1, gs), (dgr2, dgr1, dgs) = _readout_adjoint(c["wr"], c, gE.contiguous(), g.batch, T)
    d = (lambda key: c[key]) if T else (lambda key: None)
    # the seeds as a one-column Linear of four columns, whose tangent is zero
    linear("energy_head.4", g4, c["h4"], torch.zeros_like(g4) if T else None, d("dh4"), w_atom)
    linear("energy_head.2", gr2, c["h3"], dgr2, d("dh3"), w_atom)
    linear("energy_head.0", gr1, c["sL"], dgr1, d("dsL"), w_atom)
    gv = torch.zeros(n, 3, H, dtype=torch.float32, device=dev)
    if T:
        dgv = torch.zeros_like(gv)

    u = c["u"]
    if rbf_grads:
        e_mu, e_w, de_mu, de_w = _edge_feature_param_derivs(c["d"], p["rbf.centers"],
                                                           p["rbf.widths"], c["rc"])
    for k in range(L - 1, -1, -1):
        lay = c["layers"][k]
        upre = f"interactions.{k}.update"
        mpre = f"interactions.{k}.message.rbf_to_scalar"
        v_m, xin = lay["v_m"], lay["xin"]
        # update reverse (student_model.py:434-470) and its tangent
        dvm, dxin = (lay["dvm"], lay["dxin"]) if T else (None, None)
        (gy, ga2, gs_m, gv_m, gvg2), (dgy, dga2, dgs_m, dgv_m, dgvg2) = _update_adjoint(
            lay["w"], lay, gs, gv, dgs if T else None, dgv if T else None)
        linear(upre + ".update_mlp.2", gy, lay["h2"], dgy, lay["dh2"] if T else None, w_atom)
        linear(upre + ".update_mlp.0", ga2, xin, dga2, dxin, w_atom)
        if diff:
            acc(grads, upre + ".mixing_matrix",
                _xyz_outer(dgvg2, v_m, gvg2, dvm, w=w_atom, group=grp, diff=True))
        else:
            direct(upre + ".mixing_matrix", lambda: _xyz_outer(gvg2, v_m, w=w_atom, group=grp),
                   lambda: _xyz_outer(dgvg2, v_m, gvg2, dvm, group=grp))
        # message reverse (student_model.py:346-387): filter-output gradients per pair
        s, v, W = lay["s"], lay["v"], lay["W"]
        moved = (c["du"], lay["ds"], lay["dv"], dgs_m, dgv_m) if T else ()
        gW, dgW = _pair_grad(g, H, u, s, v, gs_m, gv_m, *moved)
        W1 = p[mpre + ".0.weight"]
        linear(mpre + ".2", gW, lay["h"], dgW, lay["dh"] if T else None, w_pair,
               short=False)
        # gW W2 through the SiLU (and its tangent) on the fused pair kernel
        ga1, dga1 = _filter_adjoint(p, mpre, gW, lay["a1"], dgW if T else None,
                                    lay["da1"] if T else None)
        linear(mpre + ".0", ga1, c["e"], dga1, c["de_t"] if T else None, w_pair,
               short=False)
        if rbf_grads:
            ge = ga1 @ W1
            if T:
                dge, dd = dga1 @ W1, c["dd"].unsqueeze(-1)
            for name, ek, dek in (("rbf.centers", e_mu, de_mu), ("rbf.widths", e_w, de_w)):
                direct(name, lambda: (wp(ge) * ek).sum(0),
                       lambda: (dge * ek + ge * dek * dd).sum(0))
        if k == 0:   # the first vectors are zeros: only the scalars' gradient is used
            gs, dgs = _message_adjoint_scalars(g, H, gs_m, W, dgs_m if T else None,
                                               lay["dW"] if T else None)
        elif T:
            gs, gv, dgs, dgv = _message_adjoint(g, H, gs_m, gv_m, W, dgs_m, dgv_m, lay["dW"])
        else:
            gs, gv, _, _ = _message_adjoint(g, H, gs_m, gv_m, W)
    emb_rows = p["embedding.weight"].shape[0]
    zptr, zorder = _z_segments(c["Z"], emb_rows)
    if diff:
        acc(grads, "embedding.weight", _segment_sum(zptr, wa(gs) - dgs, zorder))
    else:
        direct("embedding.weight", lambda: _segment_sum(zptr, wa(gs), zorder),
               lambda: _segment_sum(zptr, dgs, zorder))
    grp.flush()
    return grads, (tg if T and not diff else None)


# ---------------------------------------------------------------------------
# loss
# ---------------------------------------------------------------------------

def force_matching_grads(p: Dict[str, Tensor], Z: Tensor, x: Tensor, g: PairGraph, rc: float,
                         E_label: Tensor, F_label: Tensor, forces: Tensor,
                         w_energy: float = 1.0, w_force: float = 100.0,
                         rbf_grads: bool = False):
    """loss = wE MSE(E) + wF MSE(F) (train_compact_models.py:340-342) and its
    exact gradient with respect to every parameter in ``p``.  ``forces``
    are the model's forces at ``x`` (from the fused evaluation)."""
    F = forces.to(torch.float32)
    eF = F - F_label.to(torch.float32)
    dLdF = w_force * 2.0 * eF / eF.numel()
    E, cache = forward(p, Z, x, g, rc, lam=dLdF)
    B = E.shape[0]
    eE = E - E_label.to(torch.float64)
    loss = w_energy * (eE ** 2).mean() + w_force * (eF.double() ** 2).mean()
    dLdE = (w_energy * 2.0 * eE / B).to(torch.float32)
    # one reverse pass gives both parts:
    #   d/dtheta of wE MSE(E): the unit adjoint's terms weighted by dL/dE (gw)
    #   d/dtheta of wF MSE(F) = - d/dtheta < dL/dF, grad_x sum E >
    grads, _ = reverse(p, cache, g, torch.ones(B, dtype=torch.float32, device=x.device),
                       lam=dLdF, gw=dLdE, rbf_grads=rbf_grads, diff=True)
    return loss, E, F, grads


class ForceMatchingTrainer:
    """AdamW force matching on the hand-derived gradients.

    The loop mirrors the compact-student recipe
    (scripts/train_compact_models.py:302-372): loss wE MSE(E) + wF MSE(F),
    zero_grad, backward, gradient-norm clipping, optimizer step; the
    backward is force_matching_grads instead of autograd.
    """

    def __init__(self, model, lr: float = 1e-3, weight_decay: float = 0.0,
                 w_energy: float = 1.0, w_force: float = 100.0, grad_clip: float = 1.0):
        self.model = model
        self.rbf_grads = any(n.startswith("rbf.") for n, _ in model.named_parameters())
        self.w_energy, self.w_force, self.grad_clip = w_energy, w_force, grad_clip
        self.opt = torch.optim.AdamW(model.parameters(), lr=lr, weight_decay=weight_decay)
        self._p = None
        self._p_sig = None

    def _params(self) -> Dict[str, Tensor]:
        """Detached views of the model's state (the optimizer updates the
        tensors in place, so the views stay current); rebuilt when a tensor
        has been replaced (model.to(), load_state_dict(assign=True))."""
        sig = tuple(t.data_ptr() for t in self.model.parameters()) + tuple(
            t.data_ptr() for t in self.model.buffers())
        if self._p is None or sig != self._p_sig:
            self._p = {k: v.detach() for k, v in self.model.state_dict().items()}
            self._p_sig = sig
        return self._p

    def loss_and_grads(self, Z, x, sizes, E_label, F_label, cells=None, pbc=None):
        x = x.detach().to(torch.float32).contiguous()
        g = device_graph(Z, x, sizes, self.model.cutoff, cells, pbc)
        p = self._params()
        # forces of the current weights from the fused HIP evaluation.  The
        # gradient pass is enqueued behind it before its neighbour-capacity
        # check is read, so the host does not wait for the evaluation; if the
        # list overflowed, the pass runs again on the regrown evaluation.
        finish = self.model.evaluate_async(Z, x, np.asarray(sizes), cells, pbc)
        with torch.no_grad():
            res = force_matching_grads(p, Z, x, g, self.model.cutoff, E_label, F_label,
                                       finish.pending[1], self.w_energy, self.w_force,
                                       rbf_grads=self.rbf_grads)
            done = finish()
            if done is not finish.pending:
                res = force_matching_grads(p, Z, x, g, self.model.cutoff, E_label, F_label,
                                           done[1], self.w_energy, self.w_force,
                                           rbf_grads=self.rbf_grads)
        return res

    def step(self, Z, x, sizes, E_label, F_label, cells=None, pbc=None) -> float:
        loss, E, F, grads = self.loss_and_grads(Z, x, sizes, E_label, F_label, cells, pbc)
        for name, prm in self.model.named_parameters():
            gr = grads.get(name)
            prm.grad = torch.zeros_like(prm) if gr is None else gr.to(prm.dtype).reshape(prm.shape)
        if self.grad_clip and self.grad_clip > 0:
            torch.nn.utils.clip_grad_norm_(self.model.parameters(), self.grad_clip)
        self.opt.step()
        return float(loss)
