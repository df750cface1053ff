"""The FP32-arithmetic J.v where its contractions go by rows (three components,
p = 2 and 4) and where they do not, for every tangent layout and both vector
types, against the FP64 J.v of the same form: element counts that leave the
last workgroup partly filled, and both scatter modes.  Bound: FP32 products
and sums of at most 4 x 5 terms per stage, eight stages, 6e-8 each, relative
to the largest entry; the BF16 tangent is compared with itself in FP64."""
import numpy as np
import pytest

import serac_amd as sx
from serac_amd import workloads as W

pytestmark = pytest.mark.gpu
capi = sx.capi

FORMS = {"neohookean": (sx.SX_QF_NEOHOOKEAN, (1.0, 10.0, 0.25), 3), "mass_diffusion": (sx.SX_QF_MASS_DIFFUSION, (1.7, 2.1), 3),
         "j2": (sx.SX_QF_J2_LINEAR, (200.0, 0.3, 0.5, 2.0, 0.5, 1.0, 1.0), 3), "heat": (sx.SX_QF_HEAT, (1.5, 0.7), 1)}


@pytest.mark.parametrize("name", sorted(FORMS))
@pytest.mark.parametrize("p", [1, 2, 3, 4])
@pytest.mark.parametrize("scatter", [capi.SX_SCATTER_COLORED, capi.SX_SCATTER_ATOMIC])
def test_fp32_arithmetic_against_fp64(gpu_lib, name, p, scatter):
    qf, params, nc = FORMS[name]
    mesh = sx.Mesh.cuboid(5, 3, 2)
    mesh.perturb(1, 0.2)
    space = sx.Space(mesh, p, nc)
    U = sx.DeviceVector.from_numpy(W.nodal_field(space.nnodes, nc, 3, 2000, -1e-3, 1e-3))
    v = W.nodal_field(space.nnodes, nc, 4, 3000, -1.0, 1.0).astype(np.float32)
    for tangent in (capi.SX_PREC_F32, capi.SX_PREC_BF16):
        out = {}
        for arithmetic, dtype in ((capi.SX_PREC_F64, np.float64), (capi.SX_PREC_F32, np.float64),
                                  (capi.SX_PREC_F64, np.float32)):
            f = sx.Functional(space, [space])
            f.set_option(capi.SX_OPT_SCATTER, scatter)
            f.set_option(capi.SX_OPT_TANGENT_PRECISION, tangent)
            f.set_option(capi.SX_OPT_JVP_ARITHMETIC, arithmetic)
            qd = sx.QuadratureData(space.ne, (p + 1) ** 3, np.zeros(10)) if name == "j2" else None
            f.add_domain_integral(qf, params, qdata=qd)
            _, grad = f(0.0, U, wrt=0)
            out[arithmetic, dtype] = grad(sx.DeviceVector.from_numpy(v, dtype=dtype)).numpy().astype(np.float64)
        want = out.pop((capi.SX_PREC_F64, np.float64))
        for got in out.values():
            assert np.abs(got - want).max() <= 2e-6 * np.abs(want).max()
