"""The device pattern where its kernels change form: candidate lists at the sort sizes of
one wave and above what one wave sorts, incidence lists above the lanes of a group, node
counts around the chunks of the gather plan.  Integers: everything equal."""
import ctypes

import numpy as np
import pytest

from florence_amd import _lib
from oracle import df_numpy as O

pytestmark = pytest.mark.gpu


def _star(ncells, npe):
    """ncells elements that share node 0 only, their other nodes numbered from the last."""
    own = npe - 1
    el = np.zeros((ncells, npe), dtype=np.int32)
    el[:, 1:] = 1 + np.arange(ncells * own).reshape(ncells, own)[::-1]
    return el, 1 + ncells * own


def _strip(nelem, npe, overlap):
    """Elements along a line, neighbours sharing ``overlap`` nodes, in shuffled order."""
    step = npe - overlap
    el = (np.arange(nelem)[:, None] * step + np.arange(npe)[None, ::-1]).astype(np.int32)
    rng = np.random.default_rng(nelem)
    n = int(el.max()) + 1
    return rng.permutation(n).astype(np.int32)[el][rng.permutation(nelem)], n


def _device_pattern(el, nnode):
    import torch
    lib = _lib.load()
    P = _lib.ptr
    nelem, npe = el.shape
    i32 = dict(dtype=torch.int32, device="cuda")
    E = torch.as_tensor(np.ascontiguousarray(el), device="cuda")
    ep, en, np_ = torch.empty(nnode + 1, **i32), torch.empty(nelem * npe, **i32), torch.empty(nnode + 1, **i32)
    ws = torch.empty(int(lib.fl_pattern_workspace_size(nnode)), dtype=torch.uint8, device="cuda")
    nnz, deg = ctypes.c_int64(0), ctypes.c_int32(0)
    _lib.check(lib.fl_pattern_graph(P(E), nelem, npe, nnode, P(ep), P(en), P(np_), ctypes.byref(nnz),
                                    ctypes.byref(deg), P(ws), ws.numel(), _lib.stream_ptr()), "graph")
    nb = torch.empty(nnz.value, **i32)
    ip, ix = torch.empty(3 * nnode + 1, **i32), torch.empty(9 * nnz.value, **i32)
    _lib.check(lib.fl_pattern_fill(P(E), nelem, npe, nnode, P(ep), P(en), P(np_), P(nb), P(ip), P(ix),
                                   _lib.stream_ptr()), "fill")
    order = torch.empty(nnode, **i32)
    off, bd = (ctypes.c_int32 * 7)(), (ctypes.c_int32 * 6)()
    _lib.check(lib.fl_pattern_gather_plan(P(np_), nnode, P(order), off, bd, _lib.stream_ptr()), "plan")
    # the counts of another connectivity are reported
    bad = torch.full_like(np_, 0)
    rc = lib.fl_pattern_fill(P(E), nelem, npe, nnode, P(ep), P(en), P(bad), P(nb), P(torch.empty_like(ip)), None,
                             _lib.stream_ptr())
    assert rc == _lib.FL_E_ARG and b"inconsistent" in lib.fl_last_error()
    h = lambda t: t.cpu().numpy()
    return h(ep), h(en), h(np_), h(nb), h(ip), h(ix), h(order), list(off), list(bd), deg.value


@pytest.mark.parametrize("mesh", [("strip", 1, 4, 0), ("strip", 9, 10, 3), ("strip", 341, 4, 1), ("strip", 342, 4, 1),
                                  ("strip", 40, 125, 25), ("star", 16, 4), ("star", 64, 10), ("star", 65, 4),
                                  ("star", 256, 4), ("star", 257, 4), ("star", 60, 35)])
def test_pattern_equals_oracle(cuda, mesh):
    el, nnode = _strip(*mesh[1:]) if mesh[0] == "strip" else _star(*mesh[1:])
    ep, en, nptr, nb, ip, ix, order, off, bd, deg = _device_pattern(el, nnode)
    ipr, ixr = O.sparsity_pattern(el, nnode)
    assert np.array_equal(ip, ipr) and np.array_equal(ix, ixr)
    flat = el.ravel()
    assert np.array_equal(en, np.argsort(flat, kind="stable"))
    assert np.array_equal(ep, np.searchsorted(np.sort(flat), np.arange(nnode + 1)))
    d = np.diff(nptr)
    assert deg == d.max() and np.array_equal(9 * nptr, ipr[::3])
    cls = np.where(d == d.min(), 0, 1 + np.searchsorted([128, 256, 512, 1024, 2048], d))
    assert np.array_equal(order, np.argsort(cls, kind="stable"))
    assert off == [int((cls < c).sum()) for c in range(7)]
    assert bd == [int(d[cls == c].max()) if (cls == c).any() else 0 for c in range(6)]


def test_gather_plan_limit(cuda):
    el, nnode = _star(700, 4)     # node 0 has 2101 neighbours
    with pytest.raises(_lib.FlorenceAMDError, match="limit 2048"):
        _device_pattern(el, nnode)


def test_gather_plan_limit_names_the_node(cuda):
    """The error names the first node above the limit and its count.  Two centres of 700 tets
    each: nodes 5 and 3000, of 2101 neighbours."""
    a, na = _star(700, 4)
    b, nb = _star(700, 4)
    el = np.concatenate([a, b + na])
    ids = np.arange(na + nb)
    ids[[0, 5]] = [5, 0]
    ids[[na, 3000]] = [3000, na]
    with pytest.raises(_lib.FlorenceAMDError, match=r"node 5 has 2101 neighbours \(limit 2048\)"):
        _device_pattern(ids[el].astype(np.int32), na + nb)


@pytest.mark.parametrize("star", [(16, 4), (64, 10), (65, 4), (256, 4), (257, 4), (29, 35)])
def test_pattern_of_many_nodes(cuda, monkeypatch, star):
    """The stars above beside a strip that makes the mesh one of many nodes, where one wave
    takes lists of up to 1024 candidates (of few nodes: 128, the rest a workgroup a node)."""
    el, n = _star(*star)
    more, m = _strip(6200 // (star[1] - 1), star[1], 1)
    both = np.concatenate([el, more + n]).astype(np.int32)
    assert n + m > 6144
    monkeypatch.setitem(globals(), "_star", lambda *a: (both, n + m))
    test_pattern_equals_oracle(cuda, ("star",) + star)
