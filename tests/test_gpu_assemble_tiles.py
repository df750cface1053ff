"""The matrix-core assembly at the edges of its 16 x 16 node tiles and of its
groups of four points (8, 27, 64 and 125 nodes and points), for every tangent
layout, the staged and the unstaged tangent, and each stored precision: the
CSR matrix times a vector is the matrix-free J.v, and its entries, all of
them, are the oracle's.  Bounds: FP64 rounding of sums of up to 375 products."""
import numpy as np
import pytest

import oracle as O
import serac_amd as sx
from serac_amd import workloads as W

pytestmark = pytest.mark.gpu

CASES = {  # qfunctions of the two libraries, components, parameters
    "neohookean": (sx.SX_QF_NEOHOOKEAN, O.QF_NEOHOOKEAN, 3, (1.0, 10.0, 0.25)),
    "mass_diffusion": (sx.SX_QF_MASS_DIFFUSION, O.QF_MASS_DIFFUSION, 3, (1.7, 2.1)),
    "heat": (sx.SX_QF_HEAT, O.QF_HEAT, 1, (1.5, 0.7)),
    "j2": (sx.SX_QF_J2_LINEAR, O.QF_J2_LINEAR, 3, (200.0, 0.3, 0.5, 2.0, 0.5, 1.0, 1.0)),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("p", [1, 2, 3, 4])
@pytest.mark.parametrize("ordering,scatter", [(1, 0), (0, 1)])
@pytest.mark.parametrize("tangent", [sx.capi.SX_PREC_F64, sx.capi.SX_PREC_BF16])
def test_assembled_entries(gpu_lib, name, p, ordering, scatter, tangent):
    gid, oid, nc, params = CASES[name]
    gm, om = sx.Mesh.cuboid(2, 1, 1), O.Mesh.cuboid(2, 1, 1)
    gs, os_ = sx.Space(gm, p, nc, ordering), O.Space(om, p, nc, ordering)
    gf, of = sx.Functional(gs, [gs]), O.Form(os_)
    gf.set_option(sx.capi.SX_OPT_SCATTER, scatter)
    gf.set_option(sx.capi.SX_OPT_TANGENT_PRECISION, tangent)
    if name == "j2":
        qd = sx.QuadratureData(gs.ne, (p + 1) ** 3, np.zeros(10))
        gf.add_domain_integral(gid, params, qdata=qd)
        of.add_domain_integral_state(oid, params, np.zeros(10))
    else:
        gf.add_domain_integral(gid, params)
        of.add_domain_integral(oid, params)
    U = W.nodal_field(gs.nnodes, nc, 3, 2000, -0.01, 0.01, ordering)
    _, grad = gf(0.0, sx.DeviceVector.from_numpy(U), wrt=0)
    of.linearize(U)
    A = grad.assemble()
    v = W.nodal_field(gs.nnodes, nc, 4, 2000, -1.0, 1.0, ordering)
    vd, y = sx.DeviceVector.from_numpy(v), sx.DeviceVector(gs.ndof)
    A.mult(vd, y)
    jv = grad(vd).numpy()
    assert np.abs(y.numpy() - jv).max() < 1e-12 * np.abs(jv).max()
    if tangent != sx.capi.SX_PREC_F64:
        return
    K = np.zeros((gs.ndof, gs.ndof))
    emap = os_.emap()
    for e in range(gs.ne):
        d = np.concatenate([emap[e] * nc + c if ordering == 1 else c * gs.nnodes + emap[e] for c in range(nc)])
        K[np.ix_(d, d)] += of.element_matrix(0, e)
    assert np.abs(A.to_scipy().toarray() - K).max() < 1e-12 * np.abs(K).max()


@pytest.mark.parametrize("p", [2, 4])
def test_infinite_tangent_entries_stay_infinite(gpu_lib, p):
    """27 and 125 points fill the last group of four with a point that is not there: its tangent must not count.  An
    infinite mass: the middle node's function is positive at every point."""
    space = sx.Space(sx.Mesh.cuboid(1, 1, 1), p, 1)
    f = sx.Functional(space, [space])
    f.add_domain_integral(sx.SX_QF_MASS_DIFFUSION, (np.inf, 0.0))
    _, grad = f(0.0, sx.DeviceVector(space.ndof), wrt=0)
    middle = space.element_nodes()[0, space.npe // 2]
    assert grad.assemble().to_scipy()[middle, middle] == np.inf
