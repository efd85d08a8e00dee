"""Performance cases of the displacement-formulation assembler: what a user's program
has this package do, from the smallest calls to the 24^3 hex p=4 cube.

Kinds of work (``case["kind"]``):

* ``assemble``  K and T of one mesh into the reference CSR (``Assemble``, or
                ``assemble_device`` into the buffers a Newton loop keeps), FP64 or one of
                the mixed tangents;
* ``residual``  the residual-only (explicit) pass a warm start or a line search makes;
* ``solve``     one Newton step's linear solve to 1e-12 with the solver FEMSolver takes
                for the mesh (p-multigrid for hexes of p >= 2, block-Jacobi PCG otherwise);
* ``newton``    a whole ``FEMSolver.Solve``, the mesh's device plan included;
* ``batch``     one replay of the captured graph that assembles many meshes;
* ``train``     one Adam step of the warm-start network on a minibatch;
* ``predict``   the warm-start network's start for the next load increment;
* ``pattern``   the device plan of a new mesh (sparsity pattern, gather plan, tables).

Meshes are boxes of nx x ny x nz cells with edge 1/nx, jittered inside as the benchmark's
cubes are; coordinates, states, boundary data and weights come from the seed, the
topology from the case alone.
"""
import functools
import math

import numpy as np
import torch

from florence_amd import (AnisotropicMooneyRivlin_1, Assemble, AssembleResidual, BoundaryCondition,
                          DisplacementFormulation, FEMSolver, FunctionSpace, Mesh, MooneyRivlin,
                          NearlyIncompressibleMooneyRivlin, NeoHookean, QuadratureRule)
from florence_amd.assembly import DeviceMeshData, assemble_device, device_mesh_data
from florence_amd.batch import BatchedAssembly, default_rule, random_batch
from florence_amd.learned import WarmStartMLP
from florence_amd.solver import default_linear_solver, spmv
from florence_amd.workloads import clamp_and_pull, clamp_and_twist, twist_field

DEVICE = "cuda"


def listed():
    return [
        # the headline assembly: the benchmark's 24^3 cube of p=4 hexes, 6^3 Gauss-Lobatto
        # points, Mooney-Rivlin, K kept in the buffers of a Newton loop
        {"name": "assemble hex p4 24^3", "kind": "assemble", "element": "hex", "p": 4, "nx": 24, "ny": 24, "nz": 24,
         "law": "MooneyRivlin", "lobatto": True, "precision": "fp64", "csr": "fp64"},
        # the small mesh of the tet workload (3072 tets, degree-4 rule): a call of
        # Assemble where launches count
        {"name": "assemble tet p2 8^3", "kind": "assemble", "element": "tet", "p": 2, "nx": 8, "ny": 8, "nz": 8,
         "law": "NeoHookean", "lobatto": False, "precision": "fp64", "csr": "fp64"},
        # an ordinary hex mesh of odd sizes under the default Gauss rule
        {"name": "assemble hex p3 17x15x19", "kind": "assemble", "element": "hex", "p": 3, "nx": 17, "ny": 15,
         "nz": 19, "law": "MooneyRivlin", "lobatto": False, "precision": "fp64", "csr": "fp64"},
        # high-order tets: the dense contraction and the per-node sums
        {"name": "assemble tet p4 9x8x10", "kind": "assemble", "element": "tet", "p": 4, "nx": 9, "ny": 8, "nz": 10,
         "law": "NeoHookean", "lobatto": False, "precision": "fp64", "csr": "fp64"},
        # the mixed-precision Newton's tangent: FP32 contraction into FP32-stored values
        {"name": "assemble hex p4 16^3 fp32", "kind": "assemble", "element": "hex", "p": 4, "nx": 16, "ny": 16,
         "nz": 16, "law": "MooneyRivlin", "lobatto": True, "precision": "fp32", "csr": "fp32"},
        # the internal force alone, as every start of a warm-started increment is judged
        {"name": "residual hex p4 20^3", "kind": "residual", "element": "hex", "p": 4, "nx": 20, "ny": 20, "nz": 20,
         "law": "MooneyRivlin", "lobatto": True},
        # the linear solve of a Newton step on the twisted hex p=4 cube
        {"name": "solve hex p4 12^3", "kind": "solve", "element": "hex", "p": 4, "nx": 12, "ny": 12, "nz": 12,
         "law": "MooneyRivlin", "lobatto": True},
        # the whole analysis of the small tet workload, two increments of its five
        {"name": "newton tet p2 8^3", "kind": "newton", "element": "tet", "p": 2, "nx": 8, "ny": 8, "nz": 8,
         "law": "NeoHookean", "lobatto": False, "increments": 2},
        # many meshes of mixed type and order as one graph launch
        {"name": "batch 24 meshes", "kind": "batch", "meshes": 24, "mix": 3, "most": 2500},
        # the trainer's minibatch step
        {"name": "train 8192", "kind": "train", "rows": 8192},
        # the learned start of 16 members in lockstep (2^3 hex p=4 cubes, 729 nodes each)
        {"name": "predict 16 members", "kind": "predict", "members": 16},
        # a new mesh's plan
        {"name": "pattern tet p2 14x13x15", "kind": "pattern", "element": "tet", "p": 2, "nx": 14, "ny": 13,
         "nz": 15, "law": "NeoHookean", "lobatto": False},
    ]


# the most elements a drawn case of (type, p) has
MOST = {("tet", 1): 40000, ("tet", 2): 20000, ("tet", 3): 9000, ("tet", 4): 4400,
        ("hex", 1): 30000, ("hex", 2): 16000, ("hex", 3): 4900, ("hex", 4): 2600}


def _box(rng, cells):
    """nx, ny, nz of about ``cells`` cells, the sides within a factor of about two."""
    c = cells ** (1.0 / 3.0)
    return [max(1, int(round(c * math.exp(rng.uniform(-0.3, 0.3))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["assemble"] * 6 + ["residual"] * 2 + ["solve", "solve", "newton", "batch", "train", "predict",
                                                             "pattern"])
    if kind == "batch":
        return {"kind": kind, "meshes": rng.randint(5, 24), "mix": rng.randint(0, 999), "most": rng.randint(400, 2500)}
    if kind == "train":
        return {"kind": kind, "rows": 32 * int(round(math.exp(rng.uniform(math.log(8), math.log(512)))))}
    if kind == "predict":
        return {"kind": kind, "members": int(round(math.exp(rng.uniform(0.0, math.log(256)))))}
    et = rng.choice(["tet", "hex", "hex"])
    p = rng.randint(1, 4) if kind not in ("solve", "newton") or et == "tet" else rng.randint(2, 4)
    top = MOST[et, p]
    if kind == "solve":
        top = min(top, 6000 if et == "tet" else 1700)
    elif kind == "newton":
        top = min(top, 3000 if et == "tet" else 120)
    elif kind == "pattern":
        top = min(top, 16000)
    n = math.exp(rng.uniform(math.log(60.0 if et == "tet" else 8.0), math.log(top / 1.3)))
    nx, ny, nz = _box(rng, n / (6.0 if et == "tet" else 1.0))
    case = {"kind": kind, "element": et, "p": p, "nx": nx, "ny": ny, "nz": nz,
            "law": rng.choice(["NeoHookean", "MooneyRivlin"]), "lobatto": et == "hex" and p == 4 and rng.random() < 0.6}
    if kind in ("assemble", "residual") and rng.random() < 0.2:
        case["law"] = rng.choice(["NearlyIncompressibleMooneyRivlin", "AnisotropicMooneyRivlin_1"])
    if kind == "assemble":
        case["precision"], case["csr"] = rng.choice([("fp64", "fp64")] * 4 + [("fp32", "fp64"), ("fp32", "fp32"),
                                                                             ("bf16", "fp32")])
    if kind == "newton":
        case["increments"] = rng.randint(1, 2)
    return case


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=24)
def _topology(element, p, nx, ny, nz):
    """(points, elements) of the straight box mesh, cells of edge 1/nx."""
    m = Mesh()
    m.Parallelepiped((0.0, 0.0, 0.0), (1.0, ny / nx, nz / nx), nx, ny, nz, element_type=element)
    m.GetHighOrderMesh(p=p)
    return m.points, m.elements


def _mesh(case, seed):
    """The case's mesh with its inner nodes jittered by the benchmark meshes' amount."""
    points, elements = _topology(case["element"], case["p"], case["nx"], case["ny"], case["nz"])
    m = Mesh()
    m.element_type, m.points, m.elements = case["element"], points, elements
    m.InferPolynomialDegree()
    m.ChangeType()
    m.JitterInteriorNodes(0.03 / (case["nx"] * case["p"]), seed=seed)
    return m


def _rule(case):
    if case["lobatto"]:
        return QuadratureRule(qtype="lobatto", norder=case["p"] + 2, mesh_type="hex")
    return default_rule(case["element"], case["p"])


def _material(case, nelem, seed):
    law = case["law"]
    if law == "NeoHookean":
        return NeoHookean(3, mu=1.0, lamb=10.0)
    if law == "MooneyRivlin":
        return MooneyRivlin(3, mu1=0.5, mu2=0.5, lamb=20.0)
    if law == "NearlyIncompressibleMooneyRivlin":
        return NearlyIncompressibleMooneyRivlin(3, mu1=0.5, mu2=0.25, lamb=20.0)
    rng = np.random.Generator(np.random.PCG64(seed))
    n = rng.standard_normal((nelem, 3))
    return AnisotropicMooneyRivlin_1(3, mu1=0.5, mu2=0.5, mu3=0.8, lamb=20.0,
                                     anisotropic_orientations=n / np.linalg.norm(n, axis=1, keepdims=True))


def _state(X, seed):
    """A smooth deformed configuration of moderate strain."""
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    A = np.eye(3) + 0.03 * rng.uniform(-1.0, 1.0, (3, 3))
    ph = rng.uniform(0.0, 2.0 * np.pi, 3)
    return X @ A.T + 0.02 * np.sin(np.pi * X[:, [1, 2, 0]] + ph)


def _twisted(X, seed):
    """A state on the way of a twist of the x = 1 face (a tangent that is positive definite)."""
    return X + twist_field(X, np.deg2rad(2.0 + 0.3 * (seed % 17))) * X[:, [0]]


class _Solver(object):
    """What Assemble keeps its per-mesh plan on (a FEMSolver between its iterations)."""
    requires_geometry_update = True


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "predict", "batch"):
        return {"train": _prepare_train, "predict": _prepare_predict, "batch": _prepare_batch}[kind](case, seed)
    mesh = _mesh(case, seed)
    mat = _material(case, mesh.nelem, seed)
    if kind == "newton":
        form = DisplacementFormulation(mesh, quadrature_rules=_rule(case))
        bc = BoundaryCondition()
        if case["element"] == "tet":
            bc.SetDirichletCriteria(lambda: clamp_and_pull(mesh, 0.03 + 0.001 * (seed % 7)))
        else:
            bc.SetDirichletCriteria(lambda: clamp_and_twist(mesh, 3.0 + 0.1 * (seed % 7)))
        return {"case": case, "mesh": mesh, "form": form, "mat": mat, "bc": bc}
    fs = FunctionSpace(mesh, _rule(case), p=case["p"])
    if kind == "pattern":
        # numbered from another first element and another first node
        r = np.random.Generator(np.random.PCG64(seed))
        ids = np.roll(np.arange(mesh.nnode), r.integers(1, mesh.nnode))
        mesh.elements = ids[np.roll(np.asarray(mesh.elements, dtype=np.int64), r.integers(1, mesh.nelem), axis=0)]
        points = np.empty_like(mesh.points)
        points[ids] = mesh.points
        mesh.points = points
        mesh.ChangeType()
        return {"case": case, "mesh": mesh, "fs": fs}
    holder = _Solver()
    dm = device_mesh_data(holder, mesh, fs)
    xh = _twisted(mesh.points, seed) if kind == "solve" else _state(mesh.points, seed)
    x = torch.as_tensor(xh, device=DEVICE)
    st = {"case": case, "mesh": mesh, "fs": fs, "mat": mat, "holder": holder, "dm": dm, "x": x}
    if kind == "residual":
        dm.workspace(residual_only=True)
        return st
    dm.workspace()
    if kind == "assemble":
        # a Newton loop on the large or the mixed-precision tangent keeps K's buffers
        st["keep"] = case["precision"] != "fp64" or dm.nnz > 1 << 29
        if st["keep"]:
            st["V"] = torch.empty(dm.nnz, dtype=torch.float32 if case["csr"] == "fp32" else torch.float64,
                                  device=DEVICE)
            st["T"] = torch.empty(3 * dm.nnode, dtype=torch.float64, device=DEVICE)
        return st
    # solve: the first step of an increment, K at the state, the Dirichlet increment's forces
    V, _, _ = assemble_device(dm, mat, x)
    X = mesh.points
    left, right = np.abs(X[:, 0]) < 1e-10, np.abs(X[:, 0] - 1.0) < 1e-10
    uD = np.zeros_like(X)
    uD[right] = twist_field(X[right], np.deg2rad(2.0 + 0.1 * (seed % 11)))
    free = np.ones(X.shape, dtype=np.uint8)
    free[left | right] = 0
    st["free"] = torch.as_tensor(free.reshape(-1), device=DEVICE)
    rhs = torch.empty(3 * dm.nnode, dtype=torch.float64, device=DEVICE)
    spmv(dm, V, torch.as_tensor(uD.reshape(-1), device=DEVICE), rhs)
    st["rhs"] = -rhs * st["free"].to(torch.float64)
    st["V"], st["u"] = V, torch.empty_like(rhs)
    st["lin"] = default_linear_solver(dm)
    if hasattr(st["lin"], "hierarchy"):
        st["lin"].hierarchy(dm)
    return st


@functools.lru_cache(maxsize=8)
def _batch_topology(meshes, mix, most):
    return random_batch(meshes, seed=mix, nelem_range=(200, most))


def _batch(case, seed):
    """The mix's meshes with the seed's jitter, and the seed's displacement."""
    out = []
    for i, (m0, key, mat) in enumerate(_batch_topology(case["meshes"], case["mix"], case["most"])):
        m = Mesh()
        m.element_type, m.points, m.elements = m0.element_type, m0.points, m0.elements
        m.InferPolynomialDegree()
        m.ChangeType()
        h = (np.prod(np.ptp(m.points, axis=0)) / m.nelem) ** (1.0 / 3.0)
        m.JitterInteriorNodes(0.01 * h / key[1], seed=seed + i)
        out.append((m, key, mat))
    a = np.random.Generator(np.random.PCG64(seed)).uniform(0.01, 0.02, 2)
    return out, lambda X: a[0] * np.sin(np.pi * X[:, [1, 2, 0]]) + a[1] * X


def _prepare_batch(case, seed):
    meshes, disp = _batch(case, seed)
    ba = BatchedAssembly(meshes)
    ba.set_state(disp)
    ba.assemble()
    ba.capture()
    return {"case": case, "ba": ba}


def _train_inputs(case, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    n = case["rows"]
    F = torch.zeros((n, 32), device=DEVICE)
    F[:, :10] = torch.randn((n, 10), generator=g, device=DEVICE)
    T = torch.zeros((n, 32), device=DEVICE)
    T[:, :3] = torch.randn((n, 3), generator=g, device=DEVICE)
    m = 1e-3 * torch.randn(WarmStartMLP.initial_params(0).size, generator=g, device=DEVICE)
    v = 1e-6 * (0.5 + torch.rand(m.numel(), generator=g, device=DEVICE))
    return F, T, m, v


def _prepare_train(case, seed):
    """The trainer in mid-run: weights, Adam moments, a minibatch, the loop's buffers."""
    F, T, m, v = _train_inputs(case, seed)
    net = WarmStartMLP(device=DEVICE, seed=seed)
    net.m.copy_(m)
    net.v.copy_(v)
    net.step = 1000
    from florence_amd import _lib
    ws = torch.empty(int(_lib.load().fl_mlp_workspace_size(case["rows"])), dtype=torch.uint8, device=DEVICE)
    return {"case": case, "net": net, "F": F, "T": T, "ws": ws, "G": torch.empty_like(net.P),
            "loss": torch.empty(1, dtype=torch.float32, device=DEVICE)}


def _predict_inputs(case, seed):
    """Lockstep members on the 2^3 p=4 cube at increment 11 of 30: coordinates, the two
    last states, the mask and the next boundary values."""
    X0 = _topology("hex", 4, 2, 2, 2)[0]
    rng = np.random.Generator(np.random.PCG64(seed))
    n, k = case["members"], 11
    X = np.tile(X0, (n, 1))
    th, s = np.repeat(rng.uniform(0.0, 60.0, n), len(X0)), np.repeat(rng.uniform(0.8, 1.5, n), len(X0))
    inner = np.all((X > 1e-12) & (X < 1.0 - 1e-12), axis=1)
    X = X + inner[:, None] * rng.uniform(-0.03 / 8, 0.03 / 8, X.shape)

    def u(lam):
        c, sn = np.cos(np.deg2rad(th * lam) * X[:, 0]), np.sin(np.deg2rad(th * lam) * X[:, 0])
        y, z = X[:, 1] - 0.5, X[:, 2] - 0.5
        return np.stack([(s - 1.0) * lam * X[:, 0], c * y - sn * z - y, sn * y + c * z - z], axis=1)

    fixed = (np.abs(X[:, 0]) < 1e-10) | (np.abs(X[:, 0] - 1.0) < 1e-10)
    free = np.repeat((~fixed)[:, None], 3, axis=1).astype(np.uint8)
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a).reshape(-1), device=DEVICE)
    ubc = u(k / 30.0) * fixed[:, None]
    return d(X), d(u((k - 1) / 30.0)), d(u((k - 2) / 30.0)), k / 30.0, d(free), d(ubc)


def _predictor():
    import florence_amd
    import os
    return os.path.join(os.path.dirname(florence_amd.__file__), "data", "warmstart_twist_hex_p4.npz")


def _prepare_predict(case, seed):
    inp = _predict_inputs(case, seed)
    return {"case": case, "net": WarmStartMLP.load(_predictor(), device=DEVICE), "inputs": inp,
            "out": torch.empty_like(inp[0])}


# ------------------------------------------------------------------ the passes
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "assemble":
        if st["keep"]:
            V, T, _ = assemble_device(st["dm"], st["mat"], st["x"], st["V"], st["T"], precision=case["precision"],
                                      csr=case["csr"])
            return {"K": V, "T": T}
        K, T, _, _ = Assemble(st["holder"], st["fs"], None, st["mesh"], st["mat"], st["x"], None)
        return {"K": K.data, "T": T}
    if kind == "residual":
        return {"T": AssembleResidual(st["holder"], st["fs"], None, st["mesh"], st["mat"], st["x"], None)}
    if kind == "solve":
        return {"u": st["lin"].Solve(st["dm"], st["V"], st["free"], st["rhs"], st["u"])}
    if kind == "newton":
        solver = FEMSolver(optimise=True, number_of_load_increments=case["increments"], newton_raphson_tolerance=1e-8)
        res = solver.Solve(formulation=st["form"], mesh=st["mesh"], material=st["mat"], boundary_condition=st["bc"])
        return {"displacements": res.TotalDisp}
    if kind == "batch":
        st["ba"].replay()
        return {"{} p{}".format(*g["key"]): {"K": g["V"], "T": g["T"]} for g in st["ba"].groups}
    if kind == "train":
        net = st["net"]
        loss = net.train_step(st["F"], st["T"], case["rows"], 1e-3, ws=st["ws"], G=st["G"], loss=st["loss"])
        return {"loss": loss, "G": st["G"], "P": net.P, "m": net.m, "v": net.v}
    if kind == "predict":
        X, u1, u2, lam, free, ubc = st["inputs"]
        return {"u": st["net"].predict(X, u1, u2, lam, free, ubc, st["out"])}
    dm = DeviceMeshData(st["mesh"], st["fs"])
    return {"indptr": dm.indptr, "indices": dm.indices, "nbr_ptr": dm.node_nbr_ptr, "nbrs": dm.node_nbrs,
            "elem_ptr": dm.node_elem_ptr, "elem": dm.node_elem}


# ------------------------------------------------------------------ what a pass cannot do without
@functools.lru_cache(maxsize=64)
def _sizes(element, p, nx, ny, nz):
    """(elements, nodes per element, nodes, node pairs of the pattern)."""
    if element == "hex":
        pairs = 1
        for n in (nx, ny, nz):
            pairs *= n * (p + 1) ** 2 - (n - 1)
        return nx * ny * nz, (p + 1) ** 3, (nx * p + 1) * (ny * p + 1) * (nz * p + 1), pairs
    points, elements = _topology(element, p, nx, ny, nz)
    return _pattern_sizes(points, elements)


def _pattern_sizes(points, elements):
    el = np.asarray(elements, dtype=np.int64)
    keys = np.unique((el[:, :, None] * len(points) + el[:, None, :]).ravel())
    return el.shape[0], el.shape[1], len(points), keys.size


def _points(element, p, lobatto):
    if element == "tet":
        return len(default_rule("tet", p).points)
    return (p + 2 if lobatto else p + 1) ** 3


def _assembly_work(element, nelem, npe, nnode, pairs, G, vbytes):
    """Bytes: K and T written, X, x and the connectivity read.  Flops: per element the six
    distinct 3x3 blocks, sum-factorised for hexes (zeta, eta and beta contractions of the
    nine parent-gradient pairs), else the symmetric (3 npe)^2 matrix's 3G-term products."""
    if element == "hex":
        p1, q = round(npe ** (1 / 3.0)), round(G ** (1 / 3.0))
        flops = 6 * 2 * (9 * p1 ** 2 * q ** 3 + 9 * p1 ** 4 * q ** 2 + 4 * p1 ** 6 * q)
    else:
        flops = 3 * npe * (3 * npe + 1) * 3 * G
    return {"bytes": 9.0 * vbytes * pairs + 3 * 24.0 * nnode + 4.0 * nelem * npe, "flops": float(nelem) * flops}


def work(case):
    kind = case["kind"]
    if kind == "train":
        n, k = case["rows"], 32 * 128 + 128 * 128 + 128 * 32
        return {"bytes": 2 * 128.0 * n + 4.0 * 7 * k, "flops": 2.0 * n * (3 * k - 32 * 128)}
    if kind == "predict":
        n = 729 * case["members"]
        return {"bytes": n * (5 * 24.0 + 3), "flops": 2.0 * n * (10 * 128 + 128 * 128 + 128 * 3)}
    if kind == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for m, (et, p), _ in _batch_topology(case["meshes"], case["mix"], case["most"]):
            w = _assembly_work(et, *_pattern_sizes(m.points, m.elements), _points(et, p, False), 8)
            total = {k: total[k] + w[k] for k in total}
        return total
    nelem, npe, nnode, pairs = _sizes(case["element"], case["p"], case["nx"], case["ny"], case["nz"])
    G = _points(case["element"], case["p"], case["lobatto"])
    if kind == "assemble":
        return _assembly_work(case["element"], nelem, npe, nnode, pairs, G, 4 if case["csr"] == "fp32" else 8)
    if kind == "residual":
        return {"bytes": 3 * 24.0 * nnode + 4.0 * nelem * npe, "flops": 300.0 * nelem * G}
    if kind == "solve":      # the matrix, the right-hand side and the solution once
        return {"bytes": 72.0 * pairs + 48.0 * nnode, "flops": 18.0 * pairs}
    if kind == "newton":     # at least two tangents and two solves per increment
        w = _assembly_work(case["element"], nelem, npe, nnode, pairs, G, 8)
        return {"bytes": 2 * case["increments"] * (w["bytes"] + 72.0 * pairs),
                "flops": 2 * case["increments"] * (w["flops"] + 18.0 * pairs)}
    return {"bytes": 4.0 * (2 * nelem * npe + 10 * pairs + 5 * nnode), "flops": 0.0}


# ------------------------------------------------------------------ 64-bit values
def _law(name, F, J):
    """Cauchy stress and spatial tangent c_ijkl of the two laws given in closed form."""
    I = torch.eye(3, dtype=F.dtype, device=F.device)
    b = F @ F.transpose(-1, -2)
    J = J[..., None, None]
    J4 = J[..., None, None]
    ii = torch.einsum("ij,kl->ijkl", I, I)
    sym = torch.einsum("ik,jl->ijkl", I, I) + torch.einsum("il,jk->ijkl", I, I)
    if name == "NeoHookean":
        mu, lamb = 1.0, 10.0
        sig = mu / J * (b - I) + lamb * (J - 1.0) * I
        return sig, (mu / J4 - lamb * (J4 - 1.0)) * sym + lamb * (2.0 * J4 - 1.0) * ii
    m1, m2, lamb = 0.5, 0.5, 20.0
    trb = (b[..., 0, 0] + b[..., 1, 1] + b[..., 2, 2])[..., None, None]
    sig = 2.0 * m1 / J * b + 2.0 * m2 / J * (trb * b - b @ b) - 2.0 * (m1 + 2.0 * m2) / J * I + lamb * (J - 1.0) * I
    bij = b[..., :, :, None, None] * b[..., None, None, :, :]
    bik = b[..., :, None, :, None] * b[..., None, :, None, :]
    bil = b[..., :, None, None, :] * b[..., None, :, :, None]
    return sig, (2.0 * m2 / J4 * (2.0 * bij - bik - bil) + (2.0 * (m1 + 2.0 * m2) / J4 - lamb * (J4 - 1.0)) * sym
                 + lamb * (2.0 * J4 - 1.0) * ii)


def _exact_assembly(X, elements, x, Jm, w, law, tangent=True, params=None):
    """K's CSR values in the reference's order and T, in float64: the dense element
    integrals summed over the elements."""
    dev = torch.device(DEVICE)
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device=dev)
    X, x, Jm, w = f(X), x.to(torch.float64).reshape(-1, 3), f(Jm), f(np.ravel(w))
    el = torch.as_tensor(np.asarray(elements, dtype=np.int64), device=dev)
    nelem, npe = el.shape
    nnode, G = X.shape[0], w.numel()
    T = torch.zeros((nnode, 3), dtype=torch.float64, device=dev)
    chunk = max(1, int(6e7 // (9 * G * npe)))
    K = None
    if tangent:
        # position of (a, b) in the sorted node pairs; row 3a+i holds 3 deg(a) columns
        keys = torch.cat([(el[s:s + 2048, :, None] * nnode + el[s:s + 2048, None, :]).reshape(-1).unique()
                          for s in range(0, nelem, 2048)]).unique()
        ptr = torch.searchsorted(keys, torch.arange(nnode + 1, device=dev) * nnode)
        K = torch.zeros(9 * keys.numel(), dtype=torch.float64, device=dev)
        three = torch.arange(3, device=dev)
    for s in range(0, nelem, chunk):
        e = el[s:s + chunk]
        PX = torch.einsum("mag,eac->egmc", Jm, X[e])
        Px = torch.einsum("mag,eac->egmc", Jm, x[e])
        ix = torch.linalg.inv(Px)
        F = (torch.linalg.inv(PX) @ Px).transpose(-1, -2)
        J = torch.linalg.det(F)
        dV = w * torch.linalg.det(Px).abs()
        if params is None:
            sig, c = _law(law, F, J)
        else:
            sig, c = _neo_hookean(F, J, params[s:s + chunk])
        g = torch.einsum("egjm,mag->egja", ix, Jm)                      # dN_a/dx_j
        T.index_add_(0, e.reshape(-1), torch.einsum("egij,egja,eg->eai", sig, g, dV).reshape(-1, 3))
        if not tangent:
            continue
        D = c
        for i in range(3):
            D[..., i, :, i, :] += sig
        D = D * dV[..., None, None, None, None]                         # [e, g, i, j, k, l]
        pos = torch.searchsorted(keys, (e[:, :, None] * nnode + e[:, None, :]).reshape(-1)).view(-1, npe, npe)
        base = ptr[e]
        deg = (ptr[e + 1] - base)[:, :, None]
        rank = pos - base[:, :, None]
        A = g.reshape(g.shape[0], G * 3, npe).transpose(1, 2).contiguous()
        for i in range(3):
            for k in range(3):
                W = torch.einsum("egjl,egla->egja", D[:, :, i, :, k, :], g).reshape(g.shape[0], G * 3, npe)
                row = 9 * base[:, :, None] + 3 * i * deg + 3 * rank + k
                K.index_add_(0, row.reshape(-1), torch.bmm(A, W.contiguous()).reshape(-1))
    return K, T


def _neo_hookean(F, J, params):
    """Neo-Hookean stress and tangent with (mu, lamb) per element."""
    I = torch.eye(3, dtype=F.dtype, device=F.device)
    mu, lamb = params[:, 0].view(-1, 1, 1, 1), params[:, 1].view(-1, 1, 1, 1)
    b, J = F @ F.transpose(-1, -2), J[..., None, None]
    sig = mu / J * (b - I) + lamb * (J - 1.0) * I
    m4, l4, J4 = mu[..., None, None], lamb[..., None, None], J[..., None, None]
    sym = torch.einsum("ik,jl->ijkl", I, I) + torch.einsum("il,jk->ijkl", I, I)
    return sig, (m4 / J4 - l4 * (J4 - 1.0)) * sym + l4 * (2.0 * J4 - 1.0) * torch.einsum("ij,kl->ijkl", I, I)


def _exact_train(case, seed):
    F, T, m, v = (t.double() for t in _train_inputs(case, seed))
    n = case["rows"]
    P = torch.as_tensor(WarmStartMLP.initial_params(seed), device=DEVICE).double()
    s = [32 * 128, 128, 128 * 128, 128, 128 * 32, 32]
    W1, b1, W2, b2, W3, b3 = torch.split(P, s)
    W1, W2, W3 = W1.view(32, 128), W2.view(128, 128), W3.view(128, 32)
    H1 = torch.tanh(F @ W1 + b1)
    H2 = torch.tanh(H1 @ W2 + b2)
    dY = torch.zeros((n, 32), dtype=torch.float64, device=DEVICE)
    dif = (H2 @ W3 + b3 - T)[:, :3]
    dY[:, :3] = 2.0 * dif / (3 * n)
    d2 = (dY @ W3.T) * (1.0 - H2 * H2)
    d1 = (d2 @ W2.T) * (1.0 - H1 * H1)
    G = torch.cat([(F.T @ d1).reshape(-1), d1.sum(0), (H1.T @ d2).reshape(-1), d2.sum(0), (H2.T @ dY).reshape(-1),
                   dY.sum(0)])
    m = 0.9 * m + 0.1 * G
    v = 0.999 * v + 0.001 * G * G
    P = P - 1e-3 * (m / (1.0 - 0.9 ** 1001)) / (torch.sqrt(v / (1.0 - 0.999 ** 1001)) + 1e-8)
    return {"loss": (dif * dif).sum().view(1) / (3 * n), "G": G, "P": P, "m": m, "v": v}


def _exact_predict(case, seed):
    X, u1, u2, lam, free, ubc = _predict_inputs(case, seed)
    d = np.load(_predictor(), allow_pickle=False)
    f = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=DEVICE)
    W1, b1, W2, b2, W3, b3 = torch.split(f(d["P"]), [32 * 128, 128, 128 * 128, 128, 128 * 32, 32])
    norm, out = f(d["norm_in"]), f(d["norm_out"])
    v = lambda a: a.view(-1, 3)
    raw = torch.cat([v(X), v(u1), v(u1) - v(u2), torch.full_like(v(X)[:, :1], lam)], dim=1)
    H = torch.tanh(((raw - norm[:10]) * norm[10:]) @ W1.view(32, 128)[:10] + b1)
    Y = (torch.tanh(H @ W2.view(128, 128) + b2) @ W3.view(128, 32) + b3)[:, :3]
    u = 2.0 * v(u1) - v(u2) + out[:3] * Y + out[3:]
    return {"u": torch.where(free.bool(), u.reshape(-1), ubc)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "predict":
        return _exact_predict(case, seed)
    if kind == "batch":
        meshes, disp = _batch(case, seed)
        groups = {}
        for m, key, mat in meshes:
            groups.setdefault(key, []).append((m, mat))
        out = {}
        for (et, p), ms in sorted(groups.items()):
            off = np.cumsum([0] + [len(m.points) for m, _ in ms])
            X = np.concatenate([m.points for m, _ in ms])
            el = np.concatenate([np.asarray(m.elements, dtype=np.int64) + off[i] for i, (m, _) in enumerate(ms)])
            prm = np.concatenate([np.tile([[mat.mu, mat.lamb]], (m.nelem, 1)) for m, mat in ms])
            fs = FunctionSpace(ms[0][0], default_rule(et, p), p=p)
            x = torch.as_tensor(X + disp(X), device=DEVICE)
            K, T = _exact_assembly(X, el, x, fs.Jm, fs.AllGauss, "NeoHookean",
                                   params=torch.as_tensor(prm, device=DEVICE))
            out["{} p{}".format(et, p)] = {"K": K, "T": T.reshape(-1)}
        return out
    if kind not in ("assemble", "residual") or case["law"] not in ("NeoHookean", "MooneyRivlin"):
        return None
    mesh = _mesh(case, seed)
    fs = FunctionSpace(mesh, _rule(case), p=case["p"])
    x = torch.as_tensor(_state(mesh.points, seed), device=DEVICE)
    K, T = _exact_assembly(mesh.points, mesh.elements, x, fs.Jm, fs.AllGauss, case["law"], kind == "assemble")
    if kind == "residual":
        return {"T": T.reshape(-1, 1)}
    return {"K": K, "T": T.reshape(-1, 1) if case["precision"] == "fp64" and K.numel() <= 1 << 29 else T.reshape(-1)}
