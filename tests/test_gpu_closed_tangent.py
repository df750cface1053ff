"""The closed-form stored tangents against the oracle's dual-number tangents,
where the derivation could go wrong: large displacement gradients, a J2 state
that is neither symmetric nor traceless, elastic and plastic points, and both
kinematics.  Bound: FP64 rounding of the contractions, as every J.v here."""
import numpy as np
import pytest

import oracle as O
import serac_amd as sx
from serac_amd import workloads as W

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def random_field(space, seed, amp):
    return W.nodal_field(space.nnodes, 3, seed, 2000, -amp, amp, 1)


@pytest.mark.parametrize("p", [1, 4])
@pytest.mark.parametrize("geom", [0.0, 1.0])
@pytest.mark.parametrize("hardening", [(2.0, 1.5), (0.5, 0.0)])
def test_j2_with_a_general_state(gpu_lib, p, geom, hardening):
    params = (200.0, 0.3, 0.5, *hardening, 1.0, geom)
    gm, om = sx.Mesh.cuboid(2, 3, 2), O.Mesh.cuboid(2, 3, 2)
    gm.perturb(3, 0.2)
    om.perturb(3, 0.2)
    gs, os_ = sx.Space(gm, p, 3), O.Space(om, p, 3)
    nq = (p + 1) ** 3
    state = np.random.default_rng(8).uniform(-2e-3, 2e-3, (gs.ne, nq, 10))
    state[..., 9] = np.abs(state[..., 9])
    state[::2, :, :9] *= 0.1  # these elements stay elastic in part
    qd = sx.QuadratureData(gs.ne, nq, np.zeros(10))
    qd.set(state)
    gf = sx.Functional(gs, [gs])
    gf.add_domain_integral(sx.SX_QF_J2_LINEAR, params, qdata=qd)
    of = O.Form(os_)
    of.add_domain_integral_state(O.QF_J2_LINEAR, params, np.zeros(10))
    of.set_qdata(state)
    xyz = gs.node_coords()
    U = (0.02 * np.stack([xyz[:, 2], xyz[:, 0] ** 2, -0.3 * xyz[:, 1]], axis=1)).ravel() + random_field(gs, 4, 2e-4)
    r, grad = gf(0.0, sx.DeviceVector.from_numpy(U), wrt=0)
    assert relerr(r.numpy(), of.linearize(U)) < 1e-12
    dU = random_field(gs, 5, 1.0)
    assert relerr(grad(sx.DeviceVector.from_numpy(dU)).numpy(), of.jvp(dU)) < 1e-12
    assert relerr(grad.diagonal().numpy(), of.diagonal()) < 1e-12


@pytest.mark.parametrize("p", [1, 2, 3, 4])
def test_neohookean_at_large_strain(gpu_lib, p):
    gm, om = sx.Mesh.cuboid(2, 2, 3), O.Mesh.cuboid(2, 2, 3)
    gm.perturb(3, 0.2)
    om.perturb(3, 0.2)
    gs, os_ = sx.Space(gm, p, 3), O.Space(om, p, 3)
    gf, of = sx.Functional(gs, [gs]), O.Form(os_)
    gf.add_domain_integral(sx.SX_QF_NEOHOOKEAN, (1.0, 10.0, 0.25))
    of.add_domain_integral(O.QF_NEOHOOKEAN, (1.0, 10.0, 0.25))
    xyz = gs.node_coords()
    A = np.array([[0.6, 0.3, -0.2], [-0.4, -0.3, 0.1], [0.2, 0.5, 0.4]])
    U = (xyz @ A.T).ravel() + random_field(gs, 6, 1e-3)
    r, grad = gf(0.0, sx.DeviceVector.from_numpy(U), wrt=0)
    assert relerr(r.numpy(), of.linearize(U)) < 1e-12
    dU = random_field(gs, 7, 1.0)
    assert relerr(grad(sx.DeviceVector.from_numpy(dU)).numpy(), of.jvp(dU)) < 1e-12
