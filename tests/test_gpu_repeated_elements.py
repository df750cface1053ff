"""Domains that list elements more than once: every listing counts.  They run
one launch per element colour and listing with plain read-modify-writes (as
large meshes do per colour), and have to equal, bit for bit, a form whose
integrals list an element once each, which take the node sum: both add a
node's values colour by colour, listing by listing.
Cuboids with their 8 colours and meshes from arrays with greedy ones, every
order, precision and scatter order, the assembly, the shape gradient, and
plastic state against the oracle."""
import numpy as np
import pytest

import serac_amd as sx
from serac_amd import workloads as W
from test_gpu_j2 import J2_PARAMS, J2Pair, relerr

pytestmark = pytest.mark.gpu
capi = sx.capi
MATERIALS = {"neohookean": (sx.SX_QF_NEOHOOKEAN, (1.0, 10.0, 0.25), 3), "heat": (sx.SX_QF_HEAT, (1.5, 0.7), 1),
             "mass_diffusion": (sx.SX_QF_MASS_DIFFUSION, (1.7, 2.1), 3)}


def mesh_of(kind):
    if kind == "cuboid":
        mesh = sx.Mesh.cuboid(4, 3, 3)
        mesh.perturb(1, 0.2)
        return mesh
    n = np.array([4, 3, 3])
    z, y, x = (a.ravel() for a in np.meshgrid(*[np.arange(k + 1.0) / 4 for k in n[::-1]], indexing="ij"))
    e = np.array([(i, j, k) for k in range(3) for j in range(3) for i in range(4)])[np.random.default_rng(3).permutation(36)]
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    hexes = np.stack([((e[:, 2] + c[2]) * 4 + e[:, 1] + c[1]) * 5 + e[:, 0] + c[0] for c in corner], axis=1)
    return sx.Mesh.from_arrays(np.stack([x, y, z], axis=1), hexes.astype(np.int32))


def listings(ne):
    """A third of the mesh, some of it twice, some three times, mixed; and the same as lists without repetition."""
    rng = np.random.default_rng(4)
    once = rng.permutation(ne)[: ne // 3]
    twice, thrice = once[: len(once) // 2], once[: len(once) // 4]
    return rng.permutation(np.concatenate([once, twice, thrice])), [once, twice, thrice]


def results(space, material, domains, tangent, arithmetic, dtype, order):
    qf, params, nc = MATERIALS[material]
    f = sx.Functional(space, [space])
    f.set_option(capi.SX_OPT_SCATTER, capi.SX_SCATTER_COLORED)
    f.set_option(capi.SX_OPT_SCATTER_ORDER, order)
    f.set_option(capi.SX_OPT_TANGENT_PRECISION, tangent)
    f.set_option(capi.SX_OPT_JVP_ARITHMETIC, arithmetic)
    for elems in domains:
        f.add_domain_integral(qf, params, elems=elems)
    U = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, nc, 3, 2000, -1e-3, 1e-3, space.ordering))
    v = W.nodal_field(space.nnodes, nc, 4, 3000, -1.0, 1.0, space.ordering)
    out = {"residual": f(0.0, U).numpy()}
    r, grad = f(0.0, U, wrt=0)
    out["linearized residual"] = r.numpy()
    out["diagonal"] = grad.diagonal().numpy()
    out["matrix"] = grad.assemble().arrays()[2]
    out["J.v"] = grad(sx.DeviceVector.from_numpy(v, dtype=dtype)).numpy()
    if nc == 3:
        shape = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 5, 2000, -1e-2, 1e-2, space.ordering))
        f.set_shape_displacement(shape)
        _, sg = f(0.0, U, wrt="shape")
        out["shape gradient"] = sg(sx.DeviceVector.from_numpy(v)).numpy()
    return out


@pytest.mark.parametrize("kind", ["cuboid", "arrays"])
@pytest.mark.parametrize("p", [1, 2, 3, 4])
@pytest.mark.parametrize("material", list(MATERIALS))
def test_every_listing_counts(gpu_lib, kind, p, material):
    mesh = mesh_of(kind)
    for ordering in (sx.SX_ORDERING_BYNODES, sx.SX_ORDERING_BYVDIM):
        space = sx.Space(mesh, p, MATERIALS[material][2], ordering)
        repeated, once = listings(space.ne)
        for tangent, arithmetic, dtype, order in [(0, 0, np.float64, 2), (0, 0, np.float64, 1), (0, 0, np.float64, 0),
                                                  (1, 1, np.float64, 2), (2, 1, np.float64, 1), (1, 0, np.float32, 2),
                                                  (2, 0, np.float32, 0)]:
            got = results(space, material, [repeated], tangent, arithmetic, dtype, order)
            want = results(space, material, once, tangent, arithmetic, dtype, order)
            for k, b in want.items():
                assert np.isfinite(b).all() and np.abs(b).max() > 0, k
                assert np.array_equal(got[k], b), (k, tangent, arithmetic, dtype, order)


@pytest.mark.parametrize("p", [1, 2])
def test_j2_state_of_repeated_elements(gpu_lib, p):
    # every listing has its own state rows, in domain order, whatever launch its element runs in
    pr = J2Pair(3, p, J2_PARAMS["c4"], elems=[13, 2, 13, 26, 0, 14, 2, 20, 13, 9], state_seed=8)
    U = pr.shear_field(0.015, 1e-3, 14)
    pr.gf.update_qdata(True)
    R = pr.gf(0.0, sx.DeviceVector.from_numpy(U)).numpy()
    pr.of.update_qdata(True)
    assert relerr(R, pr.of.residual(U)) < 1e-12
    st, ref = pr.qd.numpy(), pr.of.qdata(nelem=pr.nel)
    assert np.abs(st - ref).max() <= 1e-12 * np.abs(ref).max()
