"""The reproducible scatter (element values, then a sum per node) against the
atomic scatter: whole meshes, domains that are a part of the mesh and listed
out of order, both orderings, every precision of the J.v, several integrals on
one form, and two threads on one form's stream.  FP64 sums of at most eight
values in another order differ by rounding, repeated calls not at all.  With
FP32 arithmetic the atomic scatter adds neighbouring elements' values in FP32
first: eight roundings of 6e-8 bound the difference."""
import threading

import numpy as np
import pytest

import serac_amd as sx
from serac_amd import workloads as W

pytestmark = pytest.mark.gpu
capi = sx.capi


def form_on(space, scatter, domains, tangent=capi.SX_PREC_F64, arithmetic=capi.SX_PREC_F64):
    f = sx.Functional(space, [space])
    f.set_option(capi.SX_OPT_SCATTER, scatter)
    f.set_option(capi.SX_OPT_TANGENT_PRECISION, tangent)
    f.set_option(capi.SX_OPT_JVP_ARITHMETIC, arithmetic)
    for k, elems in enumerate(domains):
        qf, params = [(sx.SX_QF_NEOHOOKEAN, (1.0, 10.0, 0.25)), (sx.SX_QF_MASS_DIFFUSION, (1.7, 2.1))][k]
        f.add_domain_integral(qf, params, elems=elems)
    return f


def domains_of(ne, which):
    rng = np.random.default_rng(2)
    if which == "whole":
        return [None]
    if which == "part":
        return [rng.permutation(ne)[: max(1, ne // 2)]]
    return [None, rng.permutation(ne)[: max(1, ne // 3)]]


@pytest.mark.parametrize("p", [1, 2, 3, 4])
@pytest.mark.parametrize("ordering", [0, 1])
@pytest.mark.parametrize("which", ["whole", "part", "two"])
def test_node_sum_equals_atomic(gpu_lib, p, ordering, which):
    mesh = sx.Mesh.cuboid(5, 3, 2)
    mesh.perturb(1, 0.2)
    space = sx.Space(mesh, p, 3, ordering)
    doms = domains_of(space.ne, which)
    U = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 3, 2000, -1e-3, 1e-3, ordering))
    v = W.nodal_field(space.nnodes, 3, 4, 3000, -1.0, 1.0, ordering)
    for tangent, arithmetic, dtype, tol in [(0, 0, np.float64, 1e-14), (1, 1, np.float64, 1e-6),
                                            (2, 1, np.float64, 1e-6), (1, 0, np.float32, 1e-6),
                                            (2, 0, np.float32, 1e-6)]:
        vd = sx.DeviceVector.from_numpy(v, dtype=dtype)
        got = []
        for scatter in (capi.SX_SCATTER_COLORED, capi.SX_SCATTER_ATOMIC):
            f = form_on(space, scatter, doms, tangent, arithmetic)
            r, grad = f(0.0, U, wrt=0)
            jv = sx.DeviceVector.from_numpy(np.full(space.ndof, np.nan), dtype=dtype)  # need not hold anything
            grad.mult(vd, jv)
            first = jv.numpy()
            grad.mult(vd, jv)
            if scatter == capi.SX_SCATTER_COLORED:
                assert np.array_equal(first, jv.numpy())
            got.append((r.numpy(), first, grad.diagonal().numpy()))
        for a, b, t in zip(*got, (1e-14, tol, 1e-14)):
            assert np.isfinite(a).all()
            assert np.abs(a - b).max() <= t * np.abs(b).max()


def test_two_threads_on_one_form(gpu_lib):
    space = sx.Space(sx.Mesh.cuboid(9, 8, 7), 2, 3)
    f = form_on(space, capi.SX_SCATTER_COLORED, [None])
    U = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 3, 2000, -1e-3, 1e-3))
    _, grad = f(0.0, U, wrt=0)
    vs = [sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 10 + k, 3000, -1.0, 1.0)) for k in range(2)]
    want = [grad(v).numpy() for v in vs]
    outs = [[sx.DeviceVector(space.ndof) for _ in range(20)] for _ in range(2)]

    def work(k):
        capi.call("sx_init", 0)
        for o in outs[k]:
            capi.call("sx_grad_apply", grad.h, vs[k].ptr, o.ptr)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    f.synchronize()
    for k in range(2):
        assert all(np.array_equal(o.numpy(), want[k]) for o in outs[k])


@pytest.mark.parametrize("which", ["one", "few", "all out of order"])
@pytest.mark.parametrize("ordering", [0, 1])
def test_lists_of_a_part(gpu_lib, which, ordering):
    """A domain's own node lists: a part below and one above a sixteenth of the nodes, and every node."""
    space = sx.Space(sx.Mesh.cuboid(9, 8, 7), 2, 3, ordering)
    elems = np.random.default_rng(6).permutation(space.ne)[: {"one": 1, "few": 60}.get(which)]
    U = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 3, 2000, -1e-3, 1e-3, ordering))
    v = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 4, 3000, -1.0, 1.0, ordering))
    got = []
    for scatter in (capi.SX_SCATTER_COLORED, capi.SX_SCATTER_ATOMIC):
        f = form_on(space, scatter, [elems])
        r = f(0.0, U).numpy()  # its first call: the output holds what the allocation held
        _, grad = f(0.0, U, wrt=0)
        jv = sx.DeviceVector.from_numpy(np.full(space.ndof, np.nan))
        grad.mult(v, jv)
        ess = space.boundary_dofs(0b1)
        x = sx.DeviceVector(space.ndof)
        rep = grad.cg(ess, v, x, rel_tol=1e-9, max_iter=3, raise_on_noconv=False)
        got.append((r, jv.numpy(), grad.diagonal().numpy(), rep["linear_iterations"]))
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.abs(a - b).max() <= 1e-14 * np.abs(b).max()


@pytest.mark.parametrize("nz", [67, 68])
def test_at_the_limit_of_the_element_values(gpu_lib, nz):
    """Meshes just below and just above 192 MB of element values: the sum, and the colours that large meshes take."""
    space = sx.Space(sx.Mesh.cuboid(68, 68, nz), 2, 3)
    assert (space.ne * space.npe * 3 * 8 <= 192 << 20) == (nz == 67)
    U = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 3, 2000, -1e-4, 1e-4))
    v = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, 3, 4, 3000, -1.0, 1.0))
    got = []
    for scatter in (capi.SX_SCATTER_COLORED, capi.SX_SCATTER_ATOMIC):
        f = form_on(space, scatter, [None])
        r, grad = f(0.0, U, wrt=0)
        got.append((r.numpy(), grad(v).numpy(), grad.diagonal().numpy()))
    for a, b in zip(*got):
        assert np.abs(a - b).max() <= 1e-14 * np.abs(b).max()
