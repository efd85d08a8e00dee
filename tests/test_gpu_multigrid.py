"""The p-multigrid Newton-step solver on the GPU (fl_mg_galerkin, fl_mg_pcg):

* every coarse level's operator equals the Galerkin product P^T K P of the fine
  tangent computed with scipy from the assembled CSR and the host transfer tables, to
  1e-12 relative, from both forms of point records (the factorised paths' C tensors,
  hex p=2, 3, 4; the dense path's dxi/dx and D) and by both coarse kernels (the
  factorised stiffness kernel of the coarse space, the per-point form); on the
  non-conforming 6-tet split (tet p=2) it equals the element-by-element product of the
  oracle's element matrices with each element's own p=2 -> p=1 interpolation;
* a solve meets its tolerance on the masked operator (checked by a product with the
  CSR), agrees with the block-Jacobi CG solution, and needs at least 5x fewer
  iterations on the twisted hex p=4 cube;
* FEMSolver with it reproduces the oracle's Newton solve of the twisted hex p=4 cube at n=2
  (tests/golden/newton_hex_p4_twist_cube2.npz): iteration counts and every increment's
  displacement within 1e-10, with the fine-level smoother matrix-free (the default)
  and on the CSR;
* the matrix-free tangent (fl_mf_apply, the fine smoother's operator) equals the masked
  product with the assembled CSR to 1e-13 on hexes of p = 2, 3, 4 (FP64 and FP32
  tangents: the FP32 CSR against the FP64 C records to the FP32 tangent's error), and
  two products are bitwise equal.
"""
import os

import numpy as np
import pytest
import scipy.sparse as sp

from cases import cube_mesh, deformed, function_space
from florence_amd.workloads import clamp_and_twist, cube_hex_p4, twisted_state

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")


def _csr(indptr, indices, V, n):
    return sp.csr_matrix((V.cpu().numpy().astype(np.float64), indices.cpu().numpy(), indptr.cpu().numpy()),
                         shape=(3 * n, 3 * n))


def _P(t, nfine):
    ptr, idx, w = t["P"]
    P = sp.csr_matrix((w, idx, ptr), shape=(nfine, t["fine_ids"].size))
    return sp.kron(P, sp.eye(3), format="csr")


@pytest.mark.parametrize("case", ["hex4-fp64", "hex4-fp32", "hex4-pointwise", "hex3", "hex2", "tet2"])
def test_galerkin_operators(cuda, case):
    import torch
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.multigrid import MultigridSolver, hierarchy_tables
    if case.startswith("hex4"):
        m, fs, mat = cube_hex_p4(2)
        x = twisted_state(m, 12.0)
    elif case.startswith("hex"):
        from florence_amd.materials import MooneyRivlin
        p = int(case[3])
        m = cube_mesh("hex", p, 3, jitter=0.05, seed=p)
        fs = function_space(m, p)
        mat = MooneyRivlin(3, mu1=0.5, mu2=0.5, lamb=20.0)
        x = deformed(m.points, 0.05, seed=40 + p)
    else:
        m = cube_mesh("tet", 2, 2, jitter=0.05, seed=2)
        fs = function_space(m, 2)
        from florence_amd.materials import NeoHookean
        mat = NeoHookean(3, mu=1.0, lamb=10.0)
        x = deformed(m.points, 0.04, seed=3)
    prec = "fp32" if case == "hex4-fp32" else "fp64"
    dm = DeviceMeshData(m, fs)
    V64, _, _ = assemble_device(dm, mat, x)
    K = _csr(dm.indptr, dm.indices, V64.clone(), dm.nnode)
    if prec == "fp32":
        assemble_device(dm, mat, x, precision="fp32")   # the records the Galerkin step reads
    mg = MultigridSolver()
    # hexes form the coarse operators with the factorised stiffness kernel of each coarse
    # space; "pointwise" takes the per-point form the tets use
    mg.factorised_galerkin = case != "hex4-pointwise"
    h = mg.galerkin(dm, prec)
    if case.startswith("hex"):
        assert all(lv.tensor_basis is not None for lv in h.levels)
    torch.cuda.synchronize()
    tabs = hierarchy_tables(m.element_type, m.elements, m.nnode, fs.quadrature.points)
    Kc, nf = K, m.nnode
    for lv, t in zip(h.levels, tabs):
        P = _P(t, nf)
        ref = (P.T @ Kc @ P).tocsr()
        got = _csr(lv.indptr, torch.as_tensor(_indices(lv), device="cuda"), lv.V, lv.nnode)
        if case == "tet2":
            # the 6-tet split is not conforming across the cubes' faces (neighbouring
            # tets cut a shared face along different diagonals; their p=2 face-centre
            # nodes merge), so the vertex space is not nested in the fine space and
            # the coarse operator is the element-by-element product sum_e W^T K_e W
            # of each element's own interpolation W, not P^T K P
            ew = _elementwise_coarse(m, fs, mat, x, t)
            nested = abs(ew - ref).max() / abs(ref).max()
            assert nested > 1e-3, "this mesh was expected to be non-nested"
            ref = ew
        err = abs(got - ref).max() / abs(ref).max()
        print("{} level p={}: {} nodes, |Kc - ref| / |Kc| = {:.3e}".format(case, t["degree"], lv.nnode, err),
              flush=True)
        assert err <= 1e-12, (case, t["degree"])
        assert int(lv.status[0].item()) == 0
        Kc, nf = ref, lv.nnode


def _elementwise_coarse(m, fs, mat, x, t):
    """sum_e W^T K_e W over the oracle's element matrices, W the p=2 -> p=1 tet
    interpolation of each element's own nodes."""
    from florence_amd.multigrid import coarse_basis, local_node_coordinates
    from oracle import df_numpy as O
    Ke, _ = O.element_matrices(m.points, m.elements, x, fs.Jm, fs.AllGauss, mat)
    xi = local_node_coordinates("tet", 10)
    W, _ = coarse_basis("tet", 1, xi[:4], xi)
    We = np.kron(W, np.eye(3))
    nc = t["fine_ids"].size
    rows, cols, vals = [], [], []
    for e in range(m.nelem):
        d = (3 * t["elements"][e][:, None] + np.arange(3)).ravel()
        rows.append(np.repeat(d, d.size))
        cols.append(np.tile(d, d.size))
        vals.append((We.T @ Ke[e] @ We).ravel())
    return sp.coo_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))),
                         shape=(3 * nc, 3 * nc)).tocsr()


def _indices(lv):
    """CSR column indices of a coarse level from its neighbour lists."""
    ptr = lv.node_nbr_ptr.cpu().numpy()
    nb = lv.node_nbrs.cpu().numpy()
    rows = []
    for a in range(lv.nnode):
        cols = (3 * nb[ptr[a]:ptr[a + 1]][:, None] + np.arange(3)[None, :]).ravel()
        rows += [cols] * 3
    return np.concatenate(rows).astype(np.int32)


def test_multigrid_solve_matches_block_jacobi(cuda):
    import torch
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.multigrid import MultigridSolver
    from florence_amd.solver import LinearSolver, spmv
    m, fs, mat = cube_hex_p4(3)
    dm = DeviceMeshData(m, fs)
    x = twisted_state(m, 15.0)
    V, T, _ = assemble_device(dm, mat, x)
    flags = clamp_and_twist(m, 30.0)
    free = torch.as_tensor(np.isnan(flags).ravel().astype(np.uint8), device="cuda")
    b = -(T * free.to(torch.float64))
    sols, its = {}, {}
    for name, solver in (("bj", LinearSolver(rtol=1e-10, check_every=10)), ("mg", MultigridSolver(rtol=1e-10))):
        sol = torch.zeros_like(b)
        solver.Solve(dm, V, free, b, sol)
        r = torch.empty_like(b)
        spmv(dm, V, sol, r, free)
        rel = float(torch.linalg.norm(r - b) / torch.linalg.norm(b))
        its[name] = solver.iterations[-1]
        sols[name] = sol.cpu().numpy()
        print("{}: {} iterations, |A x - b| / |b| = {:.2e}".format(name, its[name], rel), flush=True)
        assert rel <= 1.5e-10, name
    err = np.abs(sols["mg"] - sols["bj"]).max() / np.abs(sols["bj"]).max()
    print("mg vs bj solution: {:.2e}".format(err))
    assert err <= 1e-7
    assert its["mg"] * 5 <= its["bj"]
    # bitwise reproducible
    sol2 = torch.zeros_like(b)
    MultigridSolver(rtol=1e-10).Solve(dm, V, free, b, sol2)
    assert np.array_equal(sol2.cpu().numpy(), sols["mg"])


def test_multigrid_tet_and_zero_rhs(cuda):
    """The CSR-smoother path (tets: p=2 -> vertex level on the non-nested 6-tet split,
    the fine smoother on an FP32 copy of the CSR) meets its tolerance on the masked
    operator and agrees with block-Jacobi CG; a right-hand side that is 0 on every free
    dof returns x = 0 after no iteration."""
    import torch
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.materials import NeoHookean
    from florence_amd.multigrid import MultigridSolver
    from florence_amd.solver import LinearSolver, spmv
    from florence_amd.workloads import clamp_and_pull
    m = cube_mesh("tet", 2, 4, jitter=0.05, seed=4)
    fs = function_space(m, 2)
    mat = NeoHookean(3, mu=1.0, lamb=10.0)
    dm = DeviceMeshData(m, fs)
    x = deformed(m.points, 0.03, seed=5)
    V, T, _ = assemble_device(dm, mat, x)
    flags = clamp_and_pull(m)
    free = torch.as_tensor(np.isnan(flags).ravel().astype(np.uint8), device="cuda")
    b = -(T * free.to(torch.float64))
    sols = {}
    for name, solver in (("bj", LinearSolver(rtol=1e-10, check_every=10)), ("mg", MultigridSolver(rtol=1e-10))):
        sol = torch.zeros_like(b)
        solver.Solve(dm, V, free, b, sol)
        r = torch.empty_like(b)
        spmv(dm, V, sol, r, free)
        rel = float(torch.linalg.norm(r - b) / torch.linalg.norm(b))
        sols[name] = sol.cpu().numpy()
        print("tet p2 {}: {} iterations, |A x - b| / |b| = {:.2e}".format(name, solver.iterations[-1], rel),
              flush=True)
        assert rel <= 1.5e-10, name
    assert np.abs(sols["mg"] - sols["bj"]).max() <= 1e-7 * np.abs(sols["bj"]).max()
    mg = MultigridSolver(rtol=1e-10)
    zero = torch.zeros_like(b)
    sol = torch.full_like(b, 3.0)
    mg.Solve(dm, V, free, zero, sol)
    assert mg.iterations[-1] == 0 and float(sol.abs().max()) == 0.0


@pytest.mark.parametrize("case", ["hex2", "hex3", "hex4", "hex4-fp32"])
def test_matrix_free_operator(cuda, case):
    import torch
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.materials import MooneyRivlin
    from florence_amd.multigrid import matrix_free_operator, mf_apply
    from florence_amd.solver import spmv
    if case.startswith("hex4"):
        m, fs, mat = cube_hex_p4(2)
        x = twisted_state(m, 12.0)
    else:
        p = int(case[3])
        m = cube_mesh("hex", p, 3, jitter=0.05, seed=p)
        fs = function_space(m, p)
        mat = MooneyRivlin(3, mu1=0.5, mu2=0.5, lamb=20.0)
        x = deformed(m.points, 0.05, seed=30 + p)
    prec = "fp32" if case.endswith("fp32") else "fp64"
    dm = DeviceMeshData(m, fs)
    kw = {"precision": "fp32", "csr": "fp32"} if prec == "fp32" else {}
    V, _, _ = assemble_device(dm, mat, x, **kw)
    op, _ = matrix_free_operator(dm, prec)
    assert op is not None
    flags = clamp_and_twist(m, 30.0)
    free = torch.as_tensor(np.isnan(flags).ravel().astype(np.uint8), device="cuda")
    rng = np.random.default_rng(5)
    u = torch.as_tensor(rng.standard_normal(3 * m.nnode), device="cuda")
    y_csr = torch.empty_like(u)
    spmv(dm, V, u * free.to(torch.float64), y_csr, free)
    y_mf = torch.empty_like(u)
    mf_apply(dm, free, u, y_mf, prec)       # reads u as 0 on fixed dofs itself
    y2 = torch.empty_like(u)
    mf_apply(dm, free, u, y2, prec)
    torch.cuda.synchronize()
    a, b = y_mf.cpu().numpy(), y_csr.cpu().numpy()
    err = np.abs(a - b).max() / np.abs(b).max()
    print("{}: |K_mf u - K u| / |K u| = {:.2e}".format(case, err), flush=True)
    # FP32: the FP32-contracted, FP32-stored CSR against the FP64 records, the FP32
    # tangent's own error
    assert err <= (1e-5 if prec == "fp32" else 1e-13)
    assert np.all(a[free.cpu().numpy() == 0] == 0.0)
    assert np.array_equal(a, y2.cpu().numpy())


@pytest.mark.parametrize("p,n", [(1, 1), (1, 3), (2, 1), (2, 3), (3, 3), (4, 1)])
def test_matrix_free_element_groups(cuda, p, n):
    """The element kernel takes 16, 4, 2 or 1 elements a workgroup and each XCD a range of
    them: one element, and 27, which leaves workgroups in part or wholly empty.  The product
    equals the CSR's to 1e-13."""
    import torch
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.materials import NeoHookean
    from florence_amd.multigrid import mf_apply
    from florence_amd.solver import spmv
    m = cube_mesh("hex", p, n, jitter=0.05, seed=70 + p)
    dm = DeviceMeshData(m, function_space(m, p))
    V, _, _ = assemble_device(dm, NeoHookean(3, mu=1.0, lamb=10.0), deformed(m.points, 0.04, seed=71 + p))
    free = torch.ones(3 * m.nnode, dtype=torch.uint8, device="cuda")
    u = torch.as_tensor(np.sin(np.arange(3 * m.nnode) * 0.7), device="cuda")
    y, z = torch.empty_like(u), torch.empty_like(u)
    mf_apply(dm, free, u, y)
    spmv(dm, V, u, z)
    torch.cuda.synchronize()
    assert float((y - z).abs().max() / z.abs().max()) <= 1e-13


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp64-csr", "fp64-mf32", "fp64-mf64"])
def test_multigrid_newton_matches_oracle(cuda, precision):
    """fp64: the default smoother (matrix-free from BF16 copies of the C values);
    -mf32 / -mf64: from FP32 copies or the FP64 records; -csr: on the CSR values."""
    from florence_amd.boundary_condition import BoundaryCondition
    from florence_amd.multigrid import MultigridSolver
    from florence_amd.solver import FEMSolver
    ref = np.load(os.path.join(GOLD, "newton_hex_p4_twist_cube2.npz"))
    m, fs, mat = cube_hex_p4(2)

    class Form(object):
        ndim = nvar = 3
        fields = "mechanics"
        function_spaces = (fs, None, None)

    bc = BoundaryCondition()
    bc.SetDirichletCriteria(lambda mm: clamp_and_twist(mm, 30.0), m)
    kw = {"tangent_precision": "fp32", "csr_precision": "fp32"} if precision == "fp32" else {}
    solver = FEMSolver(optimise=True, number_of_load_increments=10, newton_raphson_tolerance=1e-8,
                       linear_solver=MultigridSolver(rtol=1e-12, matrix_free=precision != "fp64-csr",
                                                     smoother_records={"fp64-mf32": "fp32",
                                                                       "fp64-mf64": "fp64"}.get(precision, "bf16")),
                       **kw)
    res = solver.Solve(formulation=Form(), mesh=m, material=mat, boundary_condition=bc)
    assert not res.newton_raphson_failed_to_converge
    disp = np.moveaxis(res.TotalDisp.cpu().numpy(), 2, 0)
    errs = [np.abs(disp[k] - ref["disp"][k]).max() / np.abs(ref["disp"][k]).max() for k in range(10)]
    print("multigrid {}: newton {} (oracle {}), linear iterations {}, wall {:.3f}s, max rel err {:.2e}".format(
        precision, res.newton_iterations, ref["iterations"].tolist(), res.cg_iterations, res.wall_time, max(errs)),
        flush=True)
    if precision != "fp32":
        assert list(res.newton_iterations) == ref["iterations"].tolist()
        assert max(errs) <= 1e-10
    else:
        assert max(errs) <= 1e-8


def test_femsolver_default_linear_solver(cuda):
    """FEMSolver without a linear solver takes the multigrid for hexes of p >= 2 and
    block-Jacobi PCG for tets, and either reproduces the oracle's Newton solve (the twisted cube
    at 2^3 hexes: iterations and every increment within 1e-10)."""
    from florence_amd.boundary_condition import BoundaryCondition
    from florence_amd.multigrid import MultigridSolver
    from florence_amd.assembly import DeviceMeshData
    from florence_amd.solver import FEMSolver, LinearSolver, default_linear_solver
    ref = np.load(os.path.join(GOLD, "newton_hex_p4_twist_cube2.npz"))
    m, fs, mat = cube_hex_p4(2)

    class Form(object):
        ndim = nvar = 3
        fields = "mechanics"
        function_spaces = (fs, None, None)

    bc = BoundaryCondition()
    bc.SetDirichletCriteria(lambda mm: clamp_and_twist(mm, 30.0), m)
    solver = FEMSolver(optimise=True, number_of_load_increments=10, newton_raphson_tolerance=1e-8)
    res = solver.Solve(formulation=Form(), mesh=m, material=mat, boundary_condition=bc)
    assert isinstance(solver.linear_solver, MultigridSolver)
    assert list(res.newton_iterations) == ref["iterations"].tolist()
    disp = np.moveaxis(res.TotalDisp.cpu().numpy(), 2, 0)
    assert max(np.abs(disp[k] - ref["disp"][k]).max() / np.abs(ref["disp"][k]).max() for k in range(10)) <= 1e-10
    mt = cube_mesh("tet", 2, 1)
    assert isinstance(default_linear_solver(DeviceMeshData(mt, function_space(mt, 2))), LinearSolver)


def test_warm_spectrum_estimate_after_mask_change(cuda):
    """A lockstep solve holds converged members out of the linear solve.  After a solve
    in which only member A is free, the smoother's warm power-iteration vector lives on
    member A alone.  A warm solve in which only member B is free restricts it to B's
    dofs, finds it zero and starts the estimate again from the pseudo-random vector.
    Unrestricted, the identity rows of the held dofs pulled the estimate of lmax to about
    1, below B's spectrum, and the Chebyshev smoother diverged.  Every solve meets its
    tolerance, and the held member's update stays zero."""
    import torch
    from florence_amd.learned import LockstepNewton, TwistStretchFamily
    fam = TwistStretchFamily(n=2, nincr=4)
    ln = LockstepNewton(fam, [0, 1], forcing="fixed", linear="mg", lin_rtol=1e-10)
    u = torch.zeros(3 * ln.dm.nnode, dtype=torch.float64, device="cuda")
    ln._assemble(u)
    for live in ([True, False], [False, True], [True, True]):
        done = np.array([not v for v in live])
        g = torch.Generator(device="cuda").manual_seed(3)
        rhs = torch.randn(3 * ln.dm.nnode, dtype=torch.float64, device="cuda", generator=g) * ln.free_f
        rhs = rhs * ln._per_dof(torch.as_tensor(live, device="cuda")).to(rhs.dtype)
        du = torch.empty_like(rhs)
        ln._solve(rhs, du, done)
        r = rhs - spmv_masked(ln, du, live)
        rel = float(r.norm() / rhs.norm())
        print(live, "iterations", ln.lin.iterations[-1], "relative residual {:.1e}".format(rel), flush=True)
        assert rel <= 1e-9
        held = ~torch.as_tensor(live, device="cuda")
        assert float((du * ln._per_dof(held).to(du.dtype)).abs().max()) == 0.0


def spmv_masked(ln, x, live):
    """K x on the free dofs of the live members (the operator the held solve applies)."""
    import torch
    from florence_amd.solver import spmv
    mask = ln.free * ln._per_dof(torch.as_tensor(live, device="cuda")).to(ln.free.dtype)
    y = torch.empty_like(x)
    spmv(ln.dm, ln.V, x, y, mask)
    return y * mask.to(y.dtype)


def test_coarse_cg_in_one_launch(cuda):
    """The coarsest level's CG as one launch: the solve agrees with the launch-per-step form
    (both to 1e-12 on the residual: 1e-9 on the solution), repeats bitwise, and a coarse
    solve that gives up its first wait restarts in the launch-per-step form, bitwise."""
    import torch
    from florence_amd import _lib
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.multigrid import MultigridSolver
    m, fs, mat = cube_hex_p4(3)
    dm = DeviceMeshData(m, fs)
    V, _, _ = assemble_device(dm, mat, twisted_state(m, 5.0))
    free = torch.as_tensor(np.isnan(clamp_and_twist(m)).ravel().astype(np.uint8), device=cuda)
    b = torch.as_tensor(np.random.default_rng(0).standard_normal(free.numel()), device=cuda) * free
    lib = _lib.load()
    x = {}
    try:
        for mode in (0, 1, 2):
            _lib.check(lib.fl_set_tuning(_lib.FL_TUNE_CG, mode), "fl_set_tuning")
            x[mode] = [MultigridSolver(rtol=1e-12).Solve(dm, V, free, b, torch.empty_like(b)) for _ in range(2)]
            assert torch.equal(x[mode][0], x[mode][1])
    finally:
        lib.fl_set_tuning(_lib.FL_TUNE_CG, 0)
    assert torch.equal(x[1][0], x[2][0])
    assert float(torch.linalg.norm(x[0][0] - x[1][0]) / torch.linalg.norm(x[1][0])) <= 1e-9


@pytest.mark.parametrize("records", ["bf16", "fp32"])
def test_solve_on_a_stream_of_its_own(cuda, records):
    """Assembly and solve on another stream than the default one, which idles meanwhile: the
    smoother's rounded copy of the records is made after the assembly that writes them, so
    the solve is bitwise the default stream's.  (On any other stream the copy would be of
    the records of the state before.)"""
    import torch
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.multigrid import MultigridSolver
    m, fs, mat = cube_hex_p4(3)
    dm = DeviceMeshData(m, fs)
    x = torch.as_tensor(twisted_state(m, 12.0), device=cuda)
    x0 = torch.as_tensor(np.ascontiguousarray(m.points), device=cuda)
    free = torch.as_tensor(np.isnan(clamp_and_twist(m)).ravel().astype(np.uint8), device=cuda)
    b = torch.as_tensor(np.random.default_rng(2).standard_normal(free.numel()), device=cuda) * free

    def solve():
        V, _, _ = assemble_device(dm, mat, x)
        return MultigridSolver(rtol=1e-10, smoother_records=records).Solve(dm, V, free, b, torch.empty_like(b))

    ref = solve()
    assemble_device(dm, mat, x0)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        torch.cuda._sleep(20000000)   # the assembly starts late
        got = solve()
    s.synchronize()
    assert torch.equal(got, ref)
