"""CPU pins of the oracle: every restated function is checked against something it
did not compute itself -- the reference's tabulated data (tests/golden/
reference_tables.npz, written by tests/golden/extract_reference_tables.py), closed
forms, an independent energy formulation differentiated by torch autograd, scipy's
canonical CSR, and the second (C) restatement.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

from cases import tet_p2_cube, cube_mesh, deformed, function_space
from florence_amd.bases import (FeketePointsTet, GaussLobattoPointsHex, HexBases, NodeArrangementHex, TetBases)
from florence_amd.materials import (AnisotropicMooneyRivlin_1, LinearElastic, MooneyRivlin,
                                    NearlyIncompressibleMooneyRivlin, NeoHookean)
from florence_amd.quadrature import GaussLobattoQuadrature, QuadratureRule
from oracle import df_numpy as O
from oracle import energy as EN

GOLD = np.load(os.path.join(os.path.dirname(__file__), "golden", "reference_tables.npz"))
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ------------------------------------------------------------ tables vs reference
@pytest.mark.parametrize("n", range(2, 11))
def test_gll_matches_reference_table(n):
    z, w = GaussLobattoQuadrature(n)
    ref = GOLD["gll_{}".format(n)]
    assert np.abs(z[:, 0] - ref[:, 0]).max() < 4e-16
    assert np.abs(w[:, 0] - ref[:, 1]).max() < 4e-16
    # closed form: exact for polynomials of degree 2n-3
    for d in range(2 * n - 2):
        exact = 0.0 if d % 2 else 2.0 / (d + 1)
        assert abs((w[:, 0] * z[:, 0] ** d).sum() - exact) < 1e-14


@pytest.mark.parametrize("norder", [1, 2, 3, 4, 5, 6])
def test_tet_rules_match_reference_and_exactness(norder):
    q = QuadratureRule(norder=norder, mesh_type="tet")
    ref = GOLD["tet_quad_{}".format(norder)]
    assert np.array_equal(np.c_[q.points, q.weights], ref)
    # monomial exactness on the reference tet: int (1+x)^i (1+y)^j (1+z)^k = 2^(i+j+k+3) i! j! k! / (i+j+k+3)!
    from math import factorial
    degree = {1: 1, 2: 3, 3: 4, 4: 5, 5: 6, 6: 7}[norder]
    x = q.points + 1.0
    for i in range(degree + 1):
        for j in range(degree + 1 - i):
            for k in range(degree + 1 - i - j):
                exact = 2.0 ** (i + j + k + 3) * factorial(i) * factorial(j) * factorial(k) / factorial(i + j + k + 3)
                num = (q.weights * x[:, 0] ** i * x[:, 1] ** j * x[:, 2] ** k).sum()
                assert abs(num - exact) < 2e-13 * max(1.0, exact), (i, j, k)


@pytest.mark.parametrize("C", [0, 1, 2, 3])
def test_fekete_nodes_match_reference(C):
    assert np.array_equal(FeketePointsTet(C), GOLD["fekete_tet_{}".format(C)])


@pytest.mark.parametrize("C", [1, 2, 3, 4])
def test_hex_node_arrangement_faces(C):
    """The reference's hard-coded face tables (NodeArrangementHex(C)[0]) must list the
    local nodes that lie on each face of the element numbered by our arrangement."""
    faces = GOLD["hex_face_numbering_{}".format(C)]
    pts = GaussLobattoPointsHex(C)
    checks = [(2, -1), (2, 1), (1, -1), (1, 1), (0, -1), (0, 1)]
    for f, (axis, val) in enumerate(checks):
        on_face = set(np.where(np.abs(pts[:, axis] - val) < 1e-12)[0].tolist())
        assert set(faces[f].tolist()) == on_face
        # corners first, in the reference's order
        assert np.allclose(pts[faces[f][:4], axis], val)


# ----------------------------------------------------------------- basis pins
@pytest.mark.parametrize("C", [0, 1, 2, 3])
def test_tet_bases_kronecker_and_reproduction(C):
    p = C + 1
    nodes = FeketePointsTet(C)
    N, dN = TetBases(C, nodes, makezero_tol=0)
    assert np.abs(N - np.eye(nodes.shape[0])).max() < 1e-12
    q = QuadratureRule(norder=4, mesh_type="tet").points
    N, dN = TetBases(C, q, makezero_tol=0)
    assert np.abs(N.sum(0) - 1).max() < 1e-13
    assert np.abs(dN.sum(1)).max() < 1e-12
    # exact reproduction of a degree-p polynomial and its gradient
    f = lambda x: (x[:, 0] + 0.3) ** p - 0.5 * x[:, 1] ** max(p - 1, 0) * x[:, 2] + x[:, 2] ** p
    fx = lambda x: p * (x[:, 0] + 0.3) ** (p - 1)
    assert np.abs(N.T @ f(nodes) - f(q)).max() < 1e-12
    assert np.abs(dN[0].T @ f(nodes) - fx(q)).max() < 1e-11


@pytest.mark.parametrize("C", [0, 1, 2, 3])
def test_hex_bases_kronecker_and_reproduction(C):
    p = C + 1
    nodes = GaussLobattoPointsHex(C)
    N, _ = HexBases(C, nodes)
    assert np.abs(N - np.eye(nodes.shape[0])).max() < 1e-13
    q = QuadratureRule(norder=p + 1, mesh_type="hex").points
    N, dN = HexBases(C, q)
    f = lambda x: x[:, 0] ** p * x[:, 1] ** p * (x[:, 2] - 0.2) ** p
    fz = lambda x: p * x[:, 0] ** p * x[:, 1] ** p * (x[:, 2] - 0.2) ** (p - 1)
    assert np.abs(N.T @ f(nodes) - f(q)).max() < 1e-12
    assert np.abs(dN[2].T @ f(nodes) - fz(q)).max() < 1e-11


# --------------------------------------------------------- kinematics / materials
@pytest.mark.parametrize("et,p", [("tet", 2), ("hex", 3)])
def test_patch_affine_map(et, p):
    """x = A X + c gives F = A at every point for any p and any jitter; on unjittered
    (straight-sided) meshes sum detJ is the exact volume.  (The 6-tet split of
    neighbouring hexes does not match on shared faces, Mesh.py:8762-8766, so a jittered
    tet mesh has gaps/overlaps; curved hexes need more points for an exact volume.)"""
    A = np.array([[1.1, 0.1, 0.0], [0.05, 0.9, 0.02], [0.0, 0.03, 1.2]])
    m = cube_mesh(et, p, 2, jitter=0.05, seed=2)
    fs = function_space(m, p)
    x = m.points @ A.T + 0.3
    SG, F, detJ = O.kinematic_measures(fs.Jm, fs.AllGauss, m.points[m.elements], x[m.elements])
    assert np.abs(F - A).max() < 1e-13
    m = cube_mesh(et, p, 2)
    x = m.points @ A.T + 0.3
    _, _, detJ = O.kinematic_measures(fs.Jm, fs.AllGauss, m.points[m.elements], x[m.elements])
    assert abs(detJ.sum() - np.linalg.det(A)) < 1e-12
    _, _, detJ0 = O.kinematic_measures(fs.Jm, fs.AllGauss, m.points[m.elements], m.points[m.elements])
    assert abs(detJ0.sum() - 1.0) < 1e-12


def test_materials_at_identity():
    I = np.eye(3)[None]
    sig, H = O.neo_hookean(I, 1.3, 7.0)
    assert np.abs(sig).max() < 1e-15
    lin = lambda mu, lam: lam * np.block([[np.ones((3, 3)), np.zeros((3, 3))], [np.zeros((3, 6))]]) + \
        mu * np.diag([2, 2, 2, 1, 1, 1.0])
    assert np.abs(H[0] - lin(1.3, 7.0)).max() < 1e-14
    sig, H = O.mooney_rivlin(I, 0.5, 0.7, 20.0)
    assert np.abs(sig).max() < 1e-14
    assert np.abs(H[0] - lin(2 * 0.5 + 2 * 0.7, 20.0 + 4 * 0.7)).max() < 1e-13


def test_new_materials_at_identity():
    """sigma(I) = 0 for the three other low-level laws (any fibre direction), and the
    linear elastic tangent is LinearElastic.H_Voigt (MaterialBase.py:92-99)."""
    I = np.eye(3)[None]
    lin = lambda mu, lam: lam * np.block([[np.ones((3, 3)), np.zeros((3, 3))], [np.zeros((3, 6))]]) + \
        mu * np.diag([2, 2, 2, 1, 1, 1.0])
    sig, H = O.linear_elastic(I, 1.3, 7.0)
    assert np.abs(sig).max() == 0.0
    assert np.abs(H[0] - lin(1.3, 7.0)).max() < 1e-15
    sig, H = O.nearly_incompressible_mooney_rivlin(I, 0.6, 0.3, 15.0)
    assert np.abs(sig).max() < 1e-13
    N = np.array([0.48, -0.6, 0.64])
    sig, H = O.anisotropic_mooney_rivlin_1(I, N, 0.5, 0.4, 0.7, 20.0)
    assert np.abs(sig).max() < 1e-13


def _materials(nelem=None, seed=5):
    rng = np.random.default_rng(seed)
    ori = None
    if nelem is not None:
        ori = rng.standard_normal((nelem, 3))
        ori /= np.linalg.norm(ori, axis=1)[:, None]
    return {"NH": NeoHookean(3, mu=1.0, lamb=10.0), "MR": MooneyRivlin(3, mu1=0.5, mu2=0.5, lamb=20.0),
            "LE": LinearElastic(3, mu=1.0, lamb=10.0),
            "NIMR": NearlyIncompressibleMooneyRivlin(3, mu1=0.6, mu2=0.3, lamb=15.0),
            "AMR1": AnisotropicMooneyRivlin_1(3, mu1=0.5, mu2=0.4, mu3=0.7, lamb=20.0,
                                             anisotropic_orientations=ori)}


def test_material_tangent_symmetries():
    rng = np.random.default_rng(0)
    F = np.eye(3) + 0.2 * rng.standard_normal((5, 3, 3))
    N = rng.standard_normal((5, 3))
    for sig, H in [O.neo_hookean(F, 1.0, 10.0), O.mooney_rivlin(F, 0.5, 0.5, 20.0), O.linear_elastic(F, 1.0, 10.0),
                   O.nearly_incompressible_mooney_rivlin(F, 0.6, 0.3, 15.0),
                   O.anisotropic_mooney_rivlin_1(F, N, 0.5, 0.4, 0.7, 20.0)]:
        assert np.abs(H - np.swapaxes(H, -1, -2)).max() < 1e-12
        assert np.abs(sig - np.swapaxes(sig, -1, -2)).max() < 1e-13


# ------------------------------------------------------ energy oracle (autograd)
@pytest.mark.parametrize("et,p,qt,q", [("tet", 2, "gauss", 3), ("hex", 2, "gauss", 3), ("hex", 3, "lobatto", 5),
                                       ("tet", 3, "gauss", 4)])
@pytest.mark.parametrize("mat", ["NH", "MR", "NIMR", "AMR1"])
def test_assembly_equals_energy_derivatives(et, p, qt, q, mat):
    m = cube_mesh(et, p, 1, jitter=0.05, seed=1)
    fs = function_space(m, p, qtype=qt, norder=q)
    material = _materials(m.nelem)[mat]
    x = deformed(m.points, 0.03, seed=3)
    indptr, indices = O.sparsity_pattern(m.elements, m.nnode)
    V, T = O.assemble_csr(m.points, m.elements, x, fs.Jm, fs.AllGauss, material, indptr, indices)
    K = sp.csr_matrix((V, indices, indptr), shape=(3 * m.nnode,) * 2).toarray()
    g, Hs = EN.gradient_and_hessian(m.points, m.elements, x, fs.Jm, fs.AllGauss, material)
    assert np.abs(T - g).max() <= 1e-12 * np.abs(g).max()
    assert np.abs(K - Hs).max() <= 1e-12 * np.abs(Hs).max()


def _dense(m, fs, material, x, update=1):
    indptr, indices = O.sparsity_pattern(m.elements, m.nnode)
    V, T = O.assemble_csr(m.points, m.elements, x, fs.Jm, fs.AllGauss, material, indptr, indices,
                          requires_geometry_update=update)
    return sp.csr_matrix((V, indices, indptr), shape=(3 * m.nnode,) * 2).toarray(), T


@pytest.mark.parametrize("et,p", [("tet", 2), ("hex", 2)])
def test_linear_elastic_pins(et, p):
    """The linear elastic low-level assembler (no geometric term) is pinned by:
    * at x = X, with and without the geometry update: K is the Hessian of the
      small-strain energy sum w |det dX/dxi| (mu e:e + lamb/2 tr(e)^2), and T = 0;
    * without the update T = 0 at any x (the traction is only formed with the update,
      _ConstitutiveStiffnessDF_.h:136-148; the gradients stay those of the current
      configuration, _KinematicMeasures_.h:94-108, so K is not x-independent);
    * at a rigid rotation x = R X: K = Q K0 Q^T with Q = diag(R) per node -- an
      isotropic constitutive term rotates with the gradients, while a geometric term
      with sigma(R) != 0 would not;
    * near X: T(X + eps d) = eps K0 d + O(eps^2), which fixes the stress law (linear
      in F with sigma(I) = 0) and the traction integral."""
    m = cube_mesh(et, p, 1, jitter=0.05, seed=1)
    fs = function_space(m, p)
    mat = LinearElastic(3, mu=1.0, lamb=10.0)
    X = np.asarray(m.points)
    _, Hs = EN.gradient_and_hessian(X, m.elements, X, fs.Jm, fs.AllGauss, mat)
    scale = np.abs(Hs).max()
    K0, T0 = _dense(m, fs, mat, X, update=0)
    assert np.abs(K0 - Hs).max() <= 1e-12 * scale and np.abs(T0).max() == 0.0
    _, T0 = _dense(m, fs, mat, deformed(X, 0.05, seed=3), update=0)
    assert np.abs(T0).max() == 0.0
    K1, T1 = _dense(m, fs, mat, X, update=1)
    assert np.abs(K1 - Hs).max() <= 1e-12 * scale and np.abs(T1).max() <= 1e-14
    t = 0.4
    R = np.array([[1, 0, 0], [0, np.cos(t), -np.sin(t)], [0, np.sin(t), np.cos(t)]]) @ \
        np.array([[np.cos(0.3), 0, np.sin(0.3)], [0, 1, 0], [-np.sin(0.3), 0, np.cos(0.3)]])
    KR, _ = _dense(m, fs, mat, X @ R.T + 0.1, update=1)
    Q = np.kron(np.eye(m.nnode), R)
    assert np.abs(KR - Q @ Hs @ Q.T).max() <= 1e-12 * scale
    d = np.random.default_rng(4).standard_normal(X.shape)
    errs = []
    for eps in (1e-4, 5e-5):
        _, Te = _dense(m, fs, mat, X + eps * d, update=1)
        errs.append(np.abs(Te - eps * (Hs @ d.ravel())).max() / (eps * np.abs(Hs @ d.ravel()).max()))
    assert errs[0] < 1e-3 and 1.7 < errs[0] / errs[1] < 2.3   # first order in eps


def test_rigid_translation_and_equilibrium():
    m, fs, mat = tet_p2_cube(n=2)
    x = deformed(m.points, 0.05, seed=4)
    indptr, indices = O.sparsity_pattern(m.elements, m.nnode)
    V, T = O.assemble_csr(m.points, m.elements, x, fs.Jm, fs.AllGauss, mat, indptr, indices)
    K = sp.csr_matrix((V, indices, indptr), shape=(3 * m.nnode,) * 2)
    for d in range(3):
        u = np.zeros(3 * m.nnode)
        u[d::3] = 1.0
        assert np.abs(K @ u).max() < 1e-11 * abs(V).max()
        assert abs(T[d::3].sum()) < 1e-12 * np.abs(T).max()
    assert abs(K - K.T).max() < 1e-12 * abs(V).max()


# -------------------------------------------------------------- sparse pattern
@pytest.mark.parametrize("et,p,n", [("tet", 2, 2), ("hex", 3, 2), ("tet", 4, 1)])
def test_pattern_equals_scipy_canonical(et, p, n):
    m = cube_mesh(et, p, n)
    indptr, indices = O.sparsity_pattern(m.elements, m.nnode)
    el = np.asarray(m.elements, dtype=np.int64)
    dofs = (3 * el[:, :, None] + np.arange(3)).reshape(el.shape[0], -1)
    I = np.repeat(dofs, dofs.shape[1], axis=1).ravel()
    J = np.tile(dofs, (1, dofs.shape[1])).ravel()
    ref = sp.coo_matrix((np.ones(I.size), (I, J)), shape=(3 * m.nnode,) * 2).tocsr()
    ref.sum_duplicates()
    ref.sort_indices()
    assert np.array_equal(indptr, ref.indptr) and np.array_equal(indices, ref.indices)


# ------------------------------------------------------- second (C) restatement
def _c_oracle():
    so = os.path.join(ROOT, "oracle", "liboracle_df.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "oracle")], check=True)
    lib = ctypes.CDLL(so)
    lib.oracle_df_assemble.restype = ctypes.c_int
    return lib


def c_assemble(m, fs, mat, x, indptr, indices, update=1):
    lib = _c_oracle()
    el = np.ascontiguousarray(m.elements, dtype=np.int64)
    V = np.zeros(indices.size)
    T = np.zeros(3 * m.nnode)
    prm = np.ascontiguousarray(mat.device_parameters())
    ori = None if mat.anisotropic_orientations is None else \
        np.ascontiguousarray(mat.anisotropic_orientations, dtype=np.float64)
    P = lambda a: None if a is None else a.ctypes.data_as(ctypes.c_void_p)
    pts, xx = np.ascontiguousarray(m.points), np.ascontiguousarray(x)
    Jm, w = np.ascontiguousarray(fs.Jm), np.ascontiguousarray(fs.AllGauss.ravel())
    ip, ix = np.ascontiguousarray(indptr, dtype=np.int32), np.ascontiguousarray(indices, dtype=np.int32)
    lib.oracle_df_assemble_ex.restype = ctypes.c_int
    rc = lib.oracle_df_assemble_ex(P(pts), P(el), P(xx), P(Jm), P(w), ctypes.c_int64(fs.AllGauss.shape[0]),
                                   ctypes.c_int64(el.shape[1]), ctypes.c_int(mat.material_id), P(prm), P(ori),
                                   ctypes.c_int(update), P(ip), P(ix), P(V), P(T), ctypes.c_int64(0),
                                   ctypes.c_int64(el.shape[0]))
    assert rc == 0
    return V, T


@pytest.mark.parametrize("et,p,mat", [("tet", 2, "NH"), ("hex", 2, "MR"), ("tet", 3, "MR"), ("tet", 2, "LE"),
                                      ("hex", 2, "NIMR"), ("tet", 3, "AMR1")])
def test_c_restatement_matches_numpy(et, p, mat):
    m = cube_mesh(et, p, 2, jitter=0.05, seed=7)
    fs = function_space(m, p)
    material = _materials(m.nelem)[mat]
    x = deformed(m.points, 0.04, seed=8)
    indptr, indices = O.sparsity_pattern(m.elements, m.nnode)
    V, T = O.assemble_csr(m.points, m.elements, x, fs.Jm, fs.AllGauss, material, indptr, indices)
    Vc, Tc = c_assemble(m, fs, material, x, indptr, indices)
    assert np.abs(V - Vc).max() <= 1e-13 * np.abs(V).max()
    assert np.abs(T - Tc).max() <= 1e-13 * np.abs(T).max()


def test_oracle_translation_spread():
    """The reference algorithm's own FP64 spread, which the batch tests allow for: its
    parent gradients sum absolute coordinates (_KinematicMeasures_.h:88-89), so on a
    small-strain p=3 hex state the same oracle on the mesh translated by a quarter unit
    moves T by more than 1e-12 relative (K by far less); a long-double evaluation of
    the deformation gradient shows the FP64 value itself is that far from exact."""
    from cases import ORACLE_SHIFT, oracle_with_spread
    from florence_amd.batch import default_rule, random_batch
    from florence_amd.function_space import FunctionSpace
    batch = random_batch(14, seed=3, nelem_range=(20, 400))
    m, key, mat = batch[10]
    assert key == ("hex", 3) and m.nelem == 343
    fs = FunctionSpace(m, default_rule(*key), p=key[1])
    X = np.asarray(m.points)
    x = X + 0.02 * np.sin(np.pi * X[:, [1, 2, 0]]) + 0.01 * X
    ip, ix = O.sparsity_pattern(m.elements, m.nnode)
    (V, T, dV, dT), = oracle_with_spread([(m, fs, mat, x, ip, ix)])
    assert dT / np.abs(T).max() > 1e-12 and dV / np.abs(V).max() < 1e-13
    # translation invariance itself holds to that spread (a dropped term would not)
    assert np.abs(ORACLE_SHIFT).max() == 0.75
    # F in FP64 (reference formula) against a long-double evaluation of the same formula
    el = np.asarray(m.elements, dtype=np.int64)
    SG, F, detJ = O.kinematic_measures(fs.Jm, fs.AllGauss, X[el], x[el], 1)
    L = np.longdouble
    PGX = np.einsum("iag,eal->egil", fs.Jm.astype(L), X[el].astype(L))
    adj = np.stack([np.cross(PGX[..., 1, :], PGX[..., 2, :]), np.cross(PGX[..., 2, :], PGX[..., 0, :]),
                    np.cross(PGX[..., 0, :], PGX[..., 1, :])], axis=-1)
    iX = adj / np.einsum("...i,...i->...", PGX[..., 0, :], adj[..., :, 0])[..., None, None]
    FL = np.swapaxes(np.einsum("egja,eal->egjl", np.einsum("egjk,kag->egja", iX, fs.Jm.astype(L)),
                               x[el].astype(L)), -1, -2)
    assert np.abs(F - FL).max() > 1e-14


@pytest.mark.parametrize("p", [1, 2, 3, 4])
def test_gauss_lobatto_bases_at_many_points(p):
    """The 1D bases at an array of points are those at each point, bit for bit."""
    from florence_amd.bases import LagrangeGaussLobatto1D
    x = np.linspace(-1.0, 1.0, 7).reshape(1, 7) * np.array([[1.0], [0.3]])
    N, dN = LagrangeGaussLobatto1D(p - 1, x)
    assert N.shape == dN.shape == (p + 1, 2, 7)
    for i in np.ndindex(x.shape):
        n, dn = LagrangeGaussLobatto1D(p - 1, float(x[i]))
        assert np.array_equal(N[(slice(None),) + i], n) and np.array_equal(dN[(slice(None),) + i], dn)
