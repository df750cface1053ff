"""GPU parity for J2 plasticity with quadrature-point state (QuadratureData,
updateQdata), through the C-ABI, against the CPU oracle."""
import numpy as np
import pytest

import oracle as O
import serac_amd as sx
from serac_amd import workloads as W

pytestmark = pytest.mark.gpu

# {E, nu, sigma_y, Hi, Hk, density, geom_nonlin}
J2_PARAMS = {
    "c4": (200.0, 0.3, 0.5, 2.0, 0.0, 1.0, 1.0),
    "kinematic_small_strain": (200.0, 0.3, 0.5, 2.0, 1.5, 1.0, 0.0),
}


def relerr(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def initial_state(nelem, nq, seed):
    """A deviatoric, symmetric plastic strain and positive accumulated strain per point."""
    rng = np.random.default_rng(seed)
    A = rng.uniform(-2e-3, 2e-3, (nelem, nq, 3, 3))
    A = 0.5 * (A + np.swapaxes(A, -1, -2))
    A -= np.trace(A, axis1=-2, axis2=-1)[..., None, None] / 3 * np.eye(3)
    st = np.zeros((nelem, nq, 10))
    st[..., :9] = A.reshape(nelem, nq, 9)
    st[..., 9] = rng.uniform(0, 3e-3, (nelem, nq))
    return st


class J2Pair:
    def __init__(self, n, p, params, elems=None, perturb=0.2, scatter=0, state_seed=None):
        self.gm, self.om = sx.Mesh.cuboid(n, n, n), O.Mesh.cuboid(n, n, n)
        self.gm.perturb(42, perturb)
        self.om.perturb(42, perturb)
        self.gs, self.os = sx.Space(self.gm, p, 3, 1), O.Space(self.om, p, 3, 1)
        self.nq = (p + 1) ** 3
        nel = self.gs.ne if elems is None else len(elems)
        self.qd = sx.QuadratureData(nel, self.nq, np.zeros(10))
        self.gf = sx.Functional(self.gs, [self.gs])
        self.gf.set_option(sx.capi.SX_OPT_SCATTER, scatter)
        self.gf.add_domain_integral(sx.SX_QF_J2_LINEAR, params, elems=elems, qdata=self.qd)
        self.of = O.Form(self.os)
        self.of.add_domain_integral_state(O.QF_J2_LINEAR, params, np.zeros(10), elems)
        if state_seed is not None:
            st = initial_state(nel, self.nq, state_seed)
            self.qd.set(st)
            self.of.set_qdata(st)
        self.nel = nel

    def shear_field(self, gamma, noise, seed):
        xyz = self.gs.node_coords()
        U = np.zeros(self.gs.ndof)
        U[0::3] = gamma * xyz[:, 1] + 0.3 * gamma * xyz[:, 2] ** 2
        U[1::3] = 0.5 * gamma * xyz[:, 0] * xyz[:, 2]
        U[2::3] = -0.2 * gamma * np.sin(2 * xyz[:, 0])
        return U + W.nodal_field(self.gs.nnodes, 3, seed, 2000, -noise, noise, 1)


@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("which", ["c4", "kinematic_small_strain"])
def test_j2_residual_linearize_jvp_diag(gpu_lib, p, which):
    params = J2_PARAMS[which]
    pr = J2Pair(3, p, params, state_seed=5)
    U = pr.shear_field(0.01, 1e-3, 11)
    Ug = sx.DeviceVector.from_numpy(U)
    R = pr.gf(0.0, Ug).numpy()
    R_ref = pr.of.residual(U)
    assert np.isfinite(R).all()
    assert relerr(R, R_ref) < 1e-12
    out, grad = pr.gf(0.0, Ug, wrt=0)
    R_ref2 = pr.of.linearize(U)
    assert relerr(out.numpy(), R_ref2) < 1e-12
    # points in the plastic regime: the committed state would change
    st_before = pr.qd.numpy()
    assert np.array_equal(st_before, pr.of.qdata())  # no evaluation committed anything
    dU = W.nodal_field(pr.gs.nnodes, 3, 9, 3000, -1.0, 1.0, 1)
    jv = grad(sx.DeviceVector.from_numpy(dU)).numpy()
    jv_ref = pr.of.jvp(dU)
    assert relerr(jv, jv_ref) < 1e-12
    d = grad.diagonal().numpy()
    assert relerr(d, pr.of.diagonal()) < 1e-12


def test_j2_tangent_is_not_symmetric_with_geometric_nonlinearity(gpu_lib):
    # the full 81-entry layout is needed: <v, K w> != <w, K v> in general
    pr = J2Pair(2, 2, J2_PARAMS["c4"], state_seed=3)
    U = pr.shear_field(0.02, 1e-3, 12)
    _, grad = pr.gf(0.0, sx.DeviceVector.from_numpy(U), wrt=0)
    v = W.nodal_field(pr.gs.nnodes, 3, 1, 3000, -1, 1, 1)
    w = W.nodal_field(pr.gs.nnodes, 3, 2, 3000, -1, 1, 1)
    Kw = grad(sx.DeviceVector.from_numpy(w)).numpy()
    Kv = grad(sx.DeviceVector.from_numpy(v)).numpy()
    a, b = v @ Kw, w @ Kv
    assert abs(a - b) > 1e-8 * abs(a)
    pr.of.linearize(U)
    assert relerr(Kw, pr.of.jvp(w)) < 1e-12


@pytest.mark.parametrize("scatter", [0, 1])
def test_j2_state_commit_matches_oracle(gpu_lib, scatter):
    pr = J2Pair(3, 2, J2_PARAMS["c4"], scatter=scatter)
    U = pr.shear_field(0.01, 1e-3, 13)
    Ug = sx.DeviceVector.from_numpy(U)
    pr.gf(0.0, Ug)
    assert np.abs(pr.qd.numpy()).max() == 0.0  # no commit without updateQdata
    pr.gf.update_qdata(True)
    R = pr.gf(0.0, Ug).numpy()
    pr.gf.update_qdata(False)
    pr.of.update_qdata(True)
    R_ref = pr.of.residual(U)
    pr.of.update_qdata(False)
    assert relerr(R, R_ref) < 1e-12
    st, st_ref = pr.qd.numpy(), pr.of.qdata()
    assert st_ref[..., 9].max() > 0
    assert np.abs(st - st_ref).max() <= 1e-12 * np.abs(st_ref).max()
    # the plastic points agree on which ones yielded
    assert np.array_equal(st[..., 9] > 0, st_ref[..., 9] > 0)
    # a second committing evaluation at the same displacement changes nothing
    pr.gf.update_qdata(True)
    pr.gf(0.0, Ug)
    pr.gf.update_qdata(False)
    assert np.array_equal(pr.qd.numpy(), st)


def test_j2_domain_subset_state_rows_follow_domain_order(gpu_lib):
    # a domain listed out of element order: state rows must stay in domain order
    # (the node sum keeps slots in that order too; slots that launches permute by
    # colour are those of test_j2_state_of_repeated_elements)
    elems = [13, 2, 7, 26, 0, 14, 5, 20, 9]
    pr = J2Pair(3, 2, J2_PARAMS["c4"], elems=elems, state_seed=8)
    U = pr.shear_field(0.015, 1e-3, 14)
    Ug = sx.DeviceVector.from_numpy(U)
    pr.gf.update_qdata(True)
    R = pr.gf(0.0, Ug).numpy()
    pr.of.update_qdata(True)
    R_ref = pr.of.residual(U)
    assert relerr(R, R_ref) < 1e-12
    st, st_ref = pr.qd.numpy(), pr.of.qdata(nelem=len(elems))
    assert st.shape == (len(elems), pr.nq, 10)
    assert np.abs(st - st_ref).max() <= 1e-12 * np.abs(st_ref).max()


def test_j2_cyclic_quasistatic_matches_oracle(gpu_lib):
    # cyclic shear of the top face (z = 1) against a clamped bottom (z = 0):
    # load, reverse past zero, with the state committed after every step
    pr = J2Pair(2, 2, J2_PARAMS["c4"], perturb=0.1)
    bot = pr.gs.boundary_dofs(0b010000, 0x7)
    top = pr.gs.boundary_dofs(0b100000, 0x7)
    ess = np.union1d(bot, top).astype(np.int32)
    top_x = np.isin(ess, pr.gs.boundary_dofs(0b100000, 0x1))
    path = [0.004, 0.008, 0.004, 0.0, -0.004]
    xg = sx.DeviceVector(pr.gs.ndof)
    x = np.zeros(pr.gs.ndof)
    for g in path:
        target = np.where(top_x, g, 0.0)
        reps = sx.quasistatic_solve(pr.gf, xg, ess, target, 1, warm_start=True, rel_tol=1e-10,
                                    lin_rel_tol=1e-12, lin_max_iter=5000)
        assert reps[0]["converged"]
        # the same step on the oracle: warm start on the previous linearization
        # (du = du_bc + J^-1 (-R - J du_bc) on free rows), then Newton
        du = np.zeros_like(x)
        du[ess] = target - x[ess]
        R = pr.of.linearize(x)
        rhs = -(R + pr.of.jvp(du))
        rhs[ess] = 0.0
        d, crep = pr.of.cg(ess, rhs, rel=1e-12, maxit=5000)
        assert crep["converged"]
        x = x + d + du
        x, rep = pr.of.newton(ess, x, rel=1e-10, abs_tol=0.0, lin_rel=1e-12, lin_abs=0.0)
        assert rep["converged"]
        pr.of.update_qdata(True)
        pr.of.residual(x)
        pr.of.update_qdata(False)
        assert relerr(xg.numpy(), x) < 1e-8
        st, st_ref = pr.qd.numpy(), pr.of.qdata()
        assert np.abs(st - st_ref).max() <= 1e-8 * max(np.abs(st_ref).max(), 1e-12)
    assert pr.of.qdata()[..., 9].max() > 0  # the path yielded


def test_j2_precision_split(gpu_lib):
    pr = J2Pair(3, 2, J2_PARAMS["c4"], state_seed=4)
    U = pr.shear_field(0.01, 1e-3, 15)
    pr.gf.set_option(sx.capi.SX_OPT_TANGENT_PRECISION, sx.capi.SX_PREC_F32)
    _, grad = pr.gf(0.0, sx.DeviceVector.from_numpy(U), wrt=0)
    pr.of.linearize(U)
    dU = W.nodal_field(pr.gs.nnodes, 3, 9, 3000, -1.0, 1.0, 1)
    ref = pr.of.jvp(dU)
    jv64 = grad(sx.DeviceVector.from_numpy(dU)).numpy()
    jv32 = grad(sx.DeviceVector.from_numpy(dU.astype(np.float32), dtype=np.float32)).numpy()
    assert np.linalg.norm(jv64 - ref) / np.linalg.norm(ref) < 1e-6
    assert np.linalg.norm(jv32 - ref) / np.linalg.norm(ref) < 1e-5


def test_j2_requires_quadrature_data(gpu_lib):
    gm = sx.Mesh.cuboid(2, 2, 2)
    gs = sx.Space(gm, 1, 3, 1)
    f = sx.Functional(gs, [gs])
    with pytest.raises(sx.SeracAmdError):
        f.add_domain_integral(sx.SX_QF_J2_LINEAR, J2_PARAMS["c4"])
    with pytest.raises(sx.SeracAmdError):
        f.add_domain_integral(sx.SX_QF_J2_LINEAR, J2_PARAMS["c4"], qdata=sx.QuadratureData(7, 8, np.zeros(10)))
    with pytest.raises(sx.SeracAmdError):
        f.add_domain_integral(sx.SX_QF_NEOHOOKEAN, (1.0, 10.0, 0.25), qdata=sx.QuadratureData(8, 8, np.zeros(10)))
