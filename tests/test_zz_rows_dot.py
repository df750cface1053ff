"""Jacobi-CG with the essential rows copied inside the scalar product
(sx_cg_solve) against the copy as a launch of its own (sx_cg_solve_noalloc,
whose work memory has no mask): the same sums in the same order, so the same
bits, on one workgroup that is part full, exactly full and two, on
more entries than the reduction's grid has threads, and for lists that are
empty, unsorted or repeat a DOF.  (After the other tests: the scratch memory of
the second entry point stays allocated.)"""
import ctypes

import numpy as np
import pytest

import serac_amd as sx
from serac_amd import workloads as W

pytestmark = pytest.mark.gpu
capi = sx.capi


@pytest.mark.parametrize("cells", [(1, 1, 1), (3, 7, 7), (6, 6, 6), (64, 64, 64)])
@pytest.mark.parametrize("which", ["none", "face", "every"])
def test_rows_inside_the_dot(gpu_lib, cells, which):
    mesh = sx.Mesh.cuboid(*cells)
    space = sx.Space(mesh, 1, 1)
    f = sx.Functional(space, [space])
    f.add_domain_integral(sx.SX_QF_MASS_DIFFUSION, (1.0, 1.0))
    _, grad = f(0.0, sx.DeviceVector(space.ndof), wrt=0)
    rng = np.random.default_rng(5)
    ess = {"none": np.array([], dtype=np.int32), "face": space.boundary_dofs(0b000001, 0x1),
           "every": np.arange(space.ndof, dtype=np.int32)}[which]
    ess = rng.permutation(np.concatenate([ess, ess[:3]])).astype(np.int32)
    b = sx.DeviceVector.from_numpy(W.direction(space.nnodes, 1))
    x, y = sx.DeviceVector(space.ndof), sx.DeviceVector(space.ndof)
    rep = grad.cg(ess, b, x, rel_tol=1e-10, max_iter=40, raise_on_noconv=False)
    ref = sx.SolveReport()
    rc = capi.call_rc("sx_cg_solve_noalloc", grad.h, ess.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), len(ess),
                      b.ptr, y.ptr, 1e-10, 0.0, 40, ctypes.byref(ref))
    assert rc == (0 if rep["converged"] else capi.SX_ERR_NOCONV)
    assert rep["linear_iterations"] == ref.as_dict()["linear_iterations"] > 0
    assert np.array_equal(x.numpy(), y.numpy())
    assert np.array_equal(x.numpy()[ess], b.numpy()[ess]) or which != "every"
