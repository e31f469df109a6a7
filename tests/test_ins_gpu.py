"""Implicit advection-diffusion stage on the GPU (femx_ins_*) against the
oracle (femIncompressibleSolver's advanceAdvectionDiffusion + update,
src/femIncompressibleSolver.cpp:129-283, 471-485).

* The assembled system (CSR values after the Dirichlet rows, and the RHS)
  matches the oracle to 1e-12 of its largest entry. The GPU sums every
  entry's element contributions in the oracle's (the reference's) element
  order; the element values themselves differ only by rounding, since
  the GPU regroups them per Gauss point.
* The linear solve meets its tolerance and matches scipy's direct sparse
  solve of the oracle's system to 1e-9.
* Trajectories of several steps, with a time-dependent prescribed velocity
  and Dirichlet rows, match the oracle to 1e-9.
* The exact fixed point of the scheme (a linear field under a uniform
  velocity) holds.
* Runs are bitwise reproducible.
* Iteration caps, restarts and error paths behave as specified.
"""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from femorph_amd import meshgen
from oracle.oracle import INSOracle
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

PARAMS = dict(dt=0.02, alpha_m=0.8, alpha_f=0.6, gamma=0.7)


def _boundary(m):
    c = m.coords
    return np.where((c.min(axis=1) < 1e-12) | (c.max(axis=1) > 1 - 1e-12))[0].astype(np.int32)


def _case(kind, n, seed):
    m = meshgen.tet_cube(n, 0.15, seed) if kind == "tet" else meshgen.hex_cube(n, 0.15, seed)
    rng = np.random.default_rng(seed)
    diff = rng.uniform(0.0, 0.02, (m.n_elems, 3))
    dn = _boundary(m)
    dv = np.zeros((len(dn), 3))
    dv[:, 0] = rng.uniform(-0.1, 0.1, len(dn))
    x = m.coords
    phi = np.exp(-20.0 * ((x[:, 0] - 0.5) ** 2 + (x[:, 1] - 0.4) ** 2 + (x[:, 2] - 0.5) ** 2))
    phid = rng.normal(size=m.n_nodes) * 0.1
    return m, diff, dn, dv, phi, phid


def _pair(gpu, kind, n, seed, tol=1e-13, restart=30, max_iter=1000):
    m, diff, dn, dv, phi, phid = _case(kind, n, seed)
    g = gpu.INSSolver(gpu.DeviceMesh(m), el_diff=diff, dir_node=dn, dir_val=dv, tol=tol, max_iter=max_iter,
                      restart=restart, **PARAMS)
    o = INSOracle(m, diff, dn, dv, PARAMS["dt"], PARAMS["alpha_m"], PARAMS["alpha_f"], PARAMS["gamma"], tol=tol,
                  max_iter=max_iter, restart=restart)
    g.set_state(phi=phi, phi_dot=phid)
    o.phi, o.phid = phi.copy(), phid.copy()
    return m, g, o


@pytest.mark.parametrize("kind,n", [("tet", 5), ("hex", 4)])
def test_system_matches_oracle(gpu, kind, n):
    print("system", kind, n, flush=True)
    m, g, o = _pair(gpu, kind, n, 1)
    g.prescribe_velocity(0, 0.7)
    o.prescribe(0, 0.7)
    st = g.advdiff_solve()
    val, rhs = o.assemble()
    rp, col, gval, grhs, x = g.get_system()
    assert np.array_equal(rp, o.rp) and np.array_equal(col, o.col)
    assert np.abs(gval - val).max() <= 1e-12 * np.abs(val).max()
    assert np.abs(grhs - rhs).max() <= 1e-12 * np.abs(rhs).max()
    assert st["converged"] and st["rel_residual"] <= 1e-13
    A = sp.csr_matrix((val, o.col, o.rp), shape=(m.n_nodes, m.n_nodes)).tocsc()
    x_ref = spla.spsolve(A, rhs)
    assert rel_l2(x, x_ref) <= 1e-9, rel_l2(x, x_ref)
    _, _, vel = g.get_state()
    np.testing.assert_allclose(vel, o.vel, rtol=0, atol=1e-15)


@pytest.mark.parametrize("kind,n,vtype", [("tet", 4, 0), ("hex", 4, 1)])
def test_trajectory_matches_oracle(gpu, kind, n, vtype):
    print("trajectory", kind, n, vtype, flush=True)
    m, g, o = _pair(gpu, kind, n, 2)
    t = 0.0
    for step in range(5):
        g.prescribe_velocity(vtype, t)
        o.prescribe(vtype, t)
        st = g.advdiff_solve()
        ok, it, rr = o.advdiff_solve()
        assert st["converged"] and ok
        g.update()
        o.update()
        phi, phid, _ = g.get_state()
        assert rel_l2(phi, o.phi) <= 1e-9, (step, rel_l2(phi, o.phi))
        assert rel_l2(phid, o.phid) <= 1e-9, (step, rel_l2(phid, o.phid))
        t += PARAMS["dt"]


def test_linear_field_fixed_point(gpu):
    m = meshgen.hex_cube(4, 0.2, 3)
    u = np.array([0.4, 0.1, -0.3])
    grad = np.array([1.0, -2.0, 0.5])
    g = gpu.INSSolver(gpu.DeviceMesh(m), tol=1e-14, el_diff=np.full((m.n_elems, 3), 0.01), **PARAMS)
    c = -u @ grad
    g.set_state(phi=m.coords @ grad, phi_dot=np.full(m.n_nodes, c))
    g.prescribe_velocity(2, 0.0, np.tile(u, (m.n_nodes, 1)))
    st = g.advdiff_solve()
    assert st["converged"]
    _, _, _, _, x = g.get_system()
    np.testing.assert_allclose(x, c, rtol=1e-10)


def test_reproducible_and_restarts(gpu):
    outs = []
    for restart in (30, 30, 5):
        m, g, o = _pair(gpu, "tet", 5, 4, tol=1e-12, restart=restart)
        g.prescribe_velocity(0, 1.1)
        st = g.advdiff_solve()
        g.update()
        outs.append((g.get_state()[0], st))
    assert np.array_equal(outs[0][0], outs[1][0]) and outs[0][1] == outs[1][1]
    assert outs[2][1]["converged"] and outs[2][1]["iterations"] > 5
    assert rel_l2(outs[2][0], outs[0][0]) <= 1e-9


def test_reported_residual_on_a_large_mesh(gpu):
    """More rows than one reduction pass has blocks (> 1024 x 256): the
    solve's reductions cover every partial, so the reported relative
    residual is the true ||b - A x|| / ||b|| of the assembled system."""
    m, diff, dn, dv, phi, phid = _case("tet", 64, 7)
    assert m.n_nodes > 1024 * 256
    g = gpu.INSSolver(gpu.DeviceMesh(m), el_diff=diff, dir_node=dn, dir_val=dv, tol=1e-8, **PARAMS)
    g.set_state(phi=phi, phi_dot=phid)
    g.prescribe_velocity(0, 0.3)
    st = g.advdiff_solve()
    rp, col, val, rhs, x = g.get_system()
    A = sp.csr_matrix((val, col, rp), shape=(m.n_nodes, m.n_nodes))
    true_rel = np.linalg.norm(rhs - A @ x) / np.linalg.norm(rhs)
    assert st["converged"] and true_rel <= 1e-8
    assert abs(st["rel_residual"] / true_rel - 1.0) <= 1e-6, (st, true_rel)


def test_iteration_cap_and_errors(gpu):
    m, g, o = _pair(gpu, "tet", 4, 5, tol=1e-15, max_iter=3)
    g.prescribe_velocity(1, 0.0)
    st = g.advdiff_solve()
    assert not st["converged"] and st["iterations"] == 3 and st["rel_residual"] > 1e-15
    with pytest.raises(gpu.FemxError):
        g.prescribe_velocity(3, 0.0)
    with pytest.raises(gpu.FemxError):
        g.prescribe_velocity(2, 0.0)  # type 2 needs node velocities
    g.update()
    with pytest.raises(gpu.FemxError):
        g.update()  # no solve since the last update
    with pytest.raises(gpu.FemxError):
        gpu.INSSolver(gpu.DeviceMesh(m), restart=40, **PARAMS)
    # a zero right-hand side: zero derivative, no iterations
    z = gpu.INSSolver(gpu.DeviceMesh(m), **PARAMS)
    st = z.advdiff_solve()
    assert st["converged"] and st["iterations"] == 0
    assert not z.get_system()[4].any()


def test_system_with_long_rows(gpu):
    """tet4 rows of more entries than one pass sums in LDS (a fan's centre
    has 259), a node of no element and Dirichlet rows among them: the system
    matches the oracle to 1e-12 of its largest entry."""
    m0 = meshgen.tet_fan(3)
    m = meshgen.Mesh(np.vstack([m0.coords, [[3.0, 3.0, 3.0]]]), m0.conn)
    rng = np.random.default_rng(2)
    diff = rng.uniform(0.0, 0.02, (m.n_elems, 3))
    dn = np.arange(5, 40, 3, dtype=np.int32)
    dv = rng.normal(size=(len(dn), 3))
    vel = rng.normal(size=(m.n_nodes, 3))
    phi, phid = rng.normal(size=m.n_nodes), rng.normal(size=m.n_nodes)
    g = gpu.INSSolver(gpu.DeviceMesh(m), el_diff=diff, dir_node=dn, dir_val=dv, tol=1e-8, **PARAMS)
    o = INSOracle(m, diff, dn, dv, PARAMS["dt"], PARAMS["alpha_m"], PARAMS["alpha_f"], PARAMS["gamma"], tol=1e-8)
    g.set_state(phi=phi, phi_dot=phid, vel=vel)
    o.phi, o.phid, o.vel = phi.copy(), phid.copy(), vel.copy()
    g.advdiff_solve()
    val, rhs = o.assemble()
    rp, col, gval, grhs, _ = g.get_system()
    assert np.array_equal(rp, o.rp) and np.array_equal(col, o.col)
    assert np.diff(rp).max() > 200
    assert np.abs(gval - val).max() <= 1e-12 * np.abs(val).max()
    assert np.abs(grhs - rhs).max() <= 1e-12 * np.abs(rhs).max()


@pytest.mark.parametrize("restart", [30, 4])
@pytest.mark.parametrize("cap", range(1, 11))
def test_stop_at_every_iteration(gpu, cap, restart):
    """A solve stopped by its iteration cap, at each place where the stop can
    be found: by the next iteration's product (between the host's looks), by
    the launch before a look, at the end of a cycle; the second and third
    solves look where the first one stopped.  The iterate is the oracle's
    (n = 12: 69 workgroups of the product)."""
    m, g, o = _pair(gpu, "tet", 12, 6, tol=1e-15, restart=restart, max_iter=cap)
    g.prescribe_velocity(0, 0.4)
    o.prescribe(0, 0.4)
    _, it, rr = o.advdiff_solve()
    assert it == cap
    for _ in range(3):
        st = g.advdiff_solve()
        assert not st["converged"] and st["iterations"] == cap
        assert abs(st["rel_residual"] - rr) <= 1e-6 * rr + 1e-12, (st, rr)  # (of ||b||: the systems' rounding)
        x = g.get_system()[4]
        assert rel_l2(x, o.phid_new) <= 1e-9, rel_l2(x, o.phid_new)


def _fan(points, seed=0):
    """Tets (centre, face) over the convex hull of points on a sphere: the
    centre's row has points + 1 entries."""
    from scipy.spatial import ConvexHull
    v = np.random.default_rng(seed).normal(size=(points, 3))
    v /= np.linalg.norm(v, axis=1)[:, None]
    x = np.vstack([np.zeros(3), v])
    conn = np.hstack([np.zeros((2 * points - 4, 1), int), ConvexHull(v).simplices + 1]).astype(np.int32)
    neg = meshgen._tet_det(meshgen.Mesh(x, conn)) < 0
    conn[neg, 2], conn[neg, 3] = conn[neg, 3].copy(), conn[neg, 2].copy()
    return meshgen.Mesh(x, conn)


@pytest.mark.parametrize("points,by_rows", [(23, True), (24, True), (30, True), (47, True), (48, False), (258, False),
                                            (65538, False)])
def test_assembly_by_row_length(gpu, points, by_rows):
    """tet4 systems on both sides of the choice between the row kernel (which
    forms a row's elements once per 24 entries) and the element kernel with
    the gathers: rows of one pass, of two, too much work for one lane, and
    more entries than 16-bit places hold.  Both match the oracle to 1e-12 of
    the largest entry (the sums of the centre's row in the oracle's element
    order, or in eight lanes' partial sums)."""
    m = meshgen.tet_fan(7) if points == 65538 else _fan(points)
    assert m.n_nodes == points + 1
    rng = np.random.default_rng(points)
    diff = rng.uniform(0.0, 0.02, (m.n_elems, 3))
    dn = np.arange(2, min(points, 40), 7, dtype=np.int32)
    dv = rng.normal(size=(len(dn), 3))
    vel = rng.normal(size=(m.n_nodes, 3))
    phi, phid = rng.normal(size=m.n_nodes), rng.normal(size=m.n_nodes)
    g = gpu.INSSolver(gpu.DeviceMesh(m), el_diff=diff, dir_node=dn, dir_val=dv, tol=1e-8, max_iter=20, **PARAMS)
    o = INSOracle(m, diff, dn, dv, PARAMS["dt"], PARAMS["alpha_m"], PARAMS["alpha_f"], PARAMS["gamma"], tol=1e-8)
    g.set_state(phi=phi, phi_dot=phid, vel=vel)
    o.phi, o.phid, o.vel = phi.copy(), phid.copy(), vel.copy()
    print("rows of", points + 1, "entries", flush=True)
    g.kernel_timing(True)
    g.advdiff_solve()
    assert ("ins_rows" in g.kernel_times()) == by_rows
    val, rhs = o.assemble()
    rp, col, gval, grhs, _ = g.get_system()
    assert np.array_equal(rp, o.rp) and np.array_equal(col, o.col)
    assert np.diff(rp).max() == points + 1
    assert np.abs(gval - val).max() <= 1e-12 * np.abs(val).max()
    assert np.abs(grhs - rhs).max() <= 1e-12 * np.abs(rhs).max()


@pytest.mark.parametrize("cap", [4, 5, 8, 9, 16, 17, 31, 32, 33])
def test_iterate_of_every_basis_size(gpu, cap):
    """The Gram-Schmidt passes are kernels for bases of up to 4, 8, 16 and 32
    vectors: iterates on both sides of each border, in cycles of 32, against
    the oracle's.  (dt 5: the residual is still 6e-5 after 33 iterations.)"""
    m, diff, dn, dv, phi, phid = _case("tet", 12, 8)
    par = dict(PARAMS, dt=5.0)
    g = gpu.INSSolver(gpu.DeviceMesh(m), el_diff=diff, dir_node=dn, dir_val=dv, tol=1e-15, max_iter=cap, restart=32,
                      **par)
    o = INSOracle(m, diff, dn, dv, par["dt"], par["alpha_m"], par["alpha_f"], par["gamma"], tol=1e-15, max_iter=cap,
                  restart=32)
    g.set_state(phi=phi, phi_dot=phid)
    o.phi, o.phid = phi.copy(), phid.copy()
    g.prescribe_velocity(0, 0.4)
    o.prescribe(0, 0.4)
    _, it, rr = o.advdiff_solve()
    st = g.advdiff_solve()
    assert st["iterations"] == it == cap
    assert abs(st["rel_residual"] - rr) <= 1e-6 * rr + 1e-12, (st, rr)
    x = g.get_system()[4]
    assert rel_l2(x, o.phid_new) <= 1e-9, rel_l2(x, o.phid_new)
