"""GPU SpMV and block-Jacobi PCG against scipy on the assembled tangent of the p=2 tet cube."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from florence_amd.workloads import clamp_and_pull, cube_tet_p2

pytestmark = pytest.mark.gpu


def _setup():
    import torch
    from florence_amd.assembly import DeviceMeshData, assemble_device
    m, fs, mat = cube_tet_p2(4)
    dm = DeviceMeshData(m, fs)
    X = np.asarray(m.points)
    x = X + 0.02 * np.sin(np.pi * X[:, [1, 2, 0]])
    V, T, _ = assemble_device(dm, mat, x)
    torch.cuda.synchronize()
    K = sp.csr_matrix((V.cpu().numpy(), dm.indices.cpu().numpy(), dm.indptr.cpu().numpy()), shape=(3 * m.nnode,) * 2)
    return m, dm, V, K


def test_spmv_matches_scipy(cuda):
    import torch
    from florence_amd.solver import spmv
    m, dm, V, K = _setup()
    rng = np.random.default_rng(0)
    xv = rng.standard_normal(K.shape[0])
    x = torch.as_tensor(xv, device=cuda)
    y = torch.empty_like(x)
    spmv(dm, V, x, y)
    ref = K @ xv
    bound = 1e-14 * (abs(K) @ np.abs(xv)) + 1e-300   # summation-order bound per row
    err = np.abs(y.cpu().numpy() - ref)
    print("spmv max err {:.3e} max bound {:.3e}".format(err.max(), bound.max()), flush=True)
    assert np.all(err <= 50 * bound)
    free = np.ones(K.shape[0], dtype=np.uint8)
    free[::7] = 0
    spmv(dm, V, x, y, torch.as_tensor(free, device=cuda))
    M = sp.diags(free.astype(float))
    refm = M @ K @ M @ xv + (1 - free) * xv
    bound = 1e-14 * (abs(K) @ np.abs(xv)) + 1e-300
    assert np.all(np.abs(y.cpu().numpy() - refm) <= 50 * bound + 1e-15 * np.abs(xv))


def test_pcg_solves_reduced_system(cuda):
    import torch
    from florence_amd.solver import LinearSolver
    m, dm, V, K = _setup()
    flags = clamp_and_pull(m)
    free = np.isnan(flags.ravel()).astype(np.uint8)
    cin = np.where(free == 1)[0]
    rng = np.random.default_rng(1)
    b = rng.standard_normal(K.shape[0]) * free
    ref = np.zeros_like(b)
    ref[cin] = spla.spsolve(K[cin, :][:, cin].tocsc(), b[cin])
    ls = LinearSolver(rtol=1e-12)
    bx = torch.as_tensor(b, device=cuda)
    x = torch.zeros_like(bx)
    ls.Solve(dm, V, torch.as_tensor(free, device=cuda), bx, x)
    err = np.abs(x.cpu().numpy() - ref).max() / np.abs(ref).max()
    print("pcg iterations", ls.iterations, "rel err", err, flush=True)
    assert err < 1e-9
    assert np.all(x.cpu().numpy()[free == 0] == 0.0)


# 3x3 blocks per matrix: one workgroup; a few threads' worth each; two, four and six blocks per
# thread on the whole chip; above the one-launch form's reach
@pytest.mark.parametrize("element,p,n,csr", [("tet", 1, 1, "fp64"), ("hex", 1, 2, "fp64"), ("tet", 2, 4, "fp32"),
                                             ("tet", 2, 8, "fp64"), ("tet", 1, 17, "fp64"), ("hex", 1, 18, "fp32"),
                                             ("hex", 2, 8, "fp64"), ("hex", 2, 9, "fp64"), ("hex", 3, 9, "fp64")])
def test_pcg_in_one_launch(cuda, element, p, n, csr):
    """The one-launch CG against the launch-per-step one on the same system: both reach
    1e-10 (the true residual, by a product with the CSR, within the recursion's drift of
    it), a second solve is bitwise equal, and a solve whose first wait is given up equals
    the launch-per-step one bitwise."""
    import torch
    from cases import cube_mesh, function_space
    from florence_amd import _lib
    from florence_amd.assembly import DeviceMeshData, assemble_device
    from florence_amd.materials import NeoHookean
    from florence_amd.solver import LinearSolver, spmv
    m = cube_mesh(element, p, n, jitter=0.02, seed=n)
    dm = DeviceMeshData(m, function_space(m, p))
    V, _, _ = assemble_device(dm, NeoHookean(3, mu=1.0, lamb=10.0), m.points, precision=csr, csr=csr)
    free = np.isnan(clamp_and_pull(m).ravel()).astype(np.uint8)
    f = torch.as_tensor(free, device=cuda)
    b = torch.as_tensor(np.random.default_rng(n).standard_normal(free.size) * free, device=cuda)
    lib = _lib.load()
    x, its = {}, {}
    try:
        for mode in (0, 1, 2):
            _lib.check(lib.fl_set_tuning(_lib.FL_TUNE_CG, mode), "fl_set_tuning")
            ls = LinearSolver(rtol=1e-10, check_every=1)
            x[mode] = ls.Solve(dm, V, f, b, torch.full_like(b, float("nan"))).clone()
            again = ls.Solve(dm, V, f, b, torch.empty_like(b))
            assert torch.equal(x[mode], again)
            its[mode] = ls.iterations[0]
    finally:
        lib.fl_set_tuning(_lib.FL_TUNE_CG, 0)
    assert torch.equal(x[1], x[2]) and its[1] == its[2]
    y = torch.empty_like(b)
    for mode in (0, 1):
        spmv(dm, V, x[mode], y, f)
        rel = float(torch.linalg.norm((b - y) * f) / torch.linalg.norm(b))
        print(element, p, n, csr, "mode", mode, its[mode], "iterations, residual", rel)
        assert rel <= 1.1e-10
        assert torch.all(x[mode][f == 0] == 0)
    assert abs(its[0] - its[1]) <= max(2, its[1] // 20)


def test_pcg_zero_right_hand_side(cuda):
    import torch
    from florence_amd.solver import LinearSolver
    m, dm, V, K = _setup()
    free = torch.as_tensor(np.isnan(clamp_and_pull(m).ravel()).astype(np.uint8), device=cuda)
    ls = LinearSolver()
    x = ls.Solve(dm, V, free, torch.zeros(K.shape[0], dtype=torch.float64, device=cuda),
                 torch.full((K.shape[0],), 3.0, dtype=torch.float64, device=cuda))
    assert ls.iterations == [0] and torch.all(x == 0)


def test_pcg_in_place(cuda):
    """b and x in one array: a one-launch solve that gave up would have lost b, so the solve
    takes the launch-per-step form, bitwise (the one-launch form sums in another order)."""
    import torch
    from florence_amd import _lib
    from florence_amd.solver import LinearSolver
    m, dm, V, K = _setup()
    free = torch.as_tensor(np.isnan(clamp_and_pull(m).ravel()).astype(np.uint8), device=cuda)
    b = torch.as_tensor(np.random.default_rng(4).standard_normal(K.shape[0]), device=cuda) * free
    lib = _lib.load()
    ls = LinearSolver(rtol=1e-10)
    try:
        _lib.check(lib.fl_set_tuning(_lib.FL_TUNE_CG, 1), "fl_set_tuning")
        ref = ls.Solve(dm, V, free, b, torch.empty_like(b))
    finally:
        lib.fl_set_tuning(_lib.FL_TUNE_CG, 0)
    x = b.clone()
    ls.Solve(dm, V, free, x, x)
    assert torch.equal(x, ref)


@pytest.mark.parametrize("element,p,n,csr", [("tet", 2, 12, "fp64"), ("tet", 2, 13, "fp64"), ("tet", 3, 7, "fp64"),
                                             ("hex", 2, 10, "fp32"), ("hex", 4, 3, "fp64")])
def test_pcg_in_one_launch_largest_forms(cuda, element, p, n, csr):
    """The matrices above come to one, two and four blocks per thread in up to 63 KB of LDS.
    These come to four in 91 KB, and to five, the most there are, in 115, 88, 80 and 65 KB
    (on 256 CUs); the same checks."""
    test_pcg_in_one_launch(cuda, element, p, n, csr)
