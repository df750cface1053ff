"""Performance cases: what programs built on this framework spend their time in.

An operator case is a weak form on a hexahedral mesh, described by plain values: the mesh (elements per direction,
cuboid numbering or the shuffled numbering of a mesh read from arrays), the order, the material, the vector ordering,
the scatter mode and the precisions.  `kind` says which call is made on it:

  residual    Functional(t, U): a line search, a convergence check
  linearize   Functional(t, U, wrt=0), then the Jacobi diagonal and one J.v: the head of a Newton iteration
  jvp         Gradient.mult: the inner loop of every Krylov solve
  assemble    Gradient.assemble and one product with the matrix: handing the Jacobian to an algebraic preconditioner
  mg_solve    Gradient.mg_cg: set the multigrid hierarchy up and solve one linear system
  load_path   quasistatic_solve: warm-started load steps, Newton with Jacobi-CG
  unet        UNet.backward and UNet.adam: one training step of the learned preconditioner's network
"""
import ctypes
import math

import numpy as np
import torch

import serac_amd as sx
from serac_amd import capi

MATERIALS = {
    # name: (qfunction, parameters, components, stored tangent entries, tangent inputs per point)
    "heat": (sx.SX_QF_HEAT, (1.5, 0.7), 1, 6, 3),
    "mass_diffusion": (sx.SX_QF_MASS_DIFFUSION, (1.7, 2.1), 3, 78, 12),
    "neohookean": (sx.SX_QF_NEOHOOKEAN, (1.0, 10.0, 0.25), 3, 45, 9),
    "elastic": (sx.SX_QF_LINEAR_ELASTIC, (9.8, 0.25), 3, 45, 9),
    # E, nu, sigma_y, Hi, Hk, density, geometric nonlinearity
    "j2": (sx.SX_QF_J2_LINEAR, (200.0, 0.3, 0.5, 2.0, 0.5, 1.0, 1.0), 3, 81, 9),
}
# the state a J2 point carries from an earlier step: plastic strain (traceless) and its accumulated norm
J2_STATE = (0.002, 0.0, 0.004, 0.0, -0.001, 0.0, 0.004, 0.0, -0.001, 0.005)
PRECISION = {"f64": capi.SX_PREC_F64, "f32": capi.SX_PREC_F32, "bf16": capi.SX_PREC_BF16}
BYTES = {"f64": 8, "f32": 4, "bf16": 2}


def form_case(kind, material, order, n, *, name=None, mesh="cuboid", perturb=0.2, ordering="vdim", scatter="atomic",
              tangent="f64", arithmetic="f64", vectors="f64"):
    nx, ny, nz = n
    case = dict(kind=kind, material=material, order=order, nx=nx, ny=ny, nz=nz, mesh=mesh, perturb=perturb,
                ordering=ordering, scatter=scatter, tangent=tangent, arithmetic=arithmetic, vectors=vectors)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest configuration: a scalar heat operator on a coarse mesh, bound by launches
        form_case("jvp", "heat", 2, (16, 16, 16), name="heat_p2_16_jvp", perturb=0.0, scatter="colored"),
        # a part meshed elsewhere: first order, shuffled numbering, component-major vectors, odd sizes
        form_case("linearize", "neohookean", 1, (29, 17, 11), name="neohookean_p1_part_linearize", mesh="shuffled",
                  ordering="nodes", scatter="colored"),
        # residual evaluations of a line search, the reproducible scatter
        form_case("residual", "neohookean", 2, (57, 48, 43), name="neohookean_p2_residual", scatter="colored"),
        # the head of a Newton iteration at third order
        form_case("linearize", "neohookean", 3, (48, 40, 44), name="neohookean_p3_linearize"),
        # the same with plasticity: quadrature-point state, unsymmetric 81-entry tangent
        form_case("linearize", "j2", 2, (56, 48, 50), name="j2_p2_linearize", perturb=0.0),
        # the headline operator: J.v in FP64
        form_case("jvp", "neohookean", 3, (64, 64, 64), name="neohookean_p3_64_jvp"),
        # fourth order in a mixed-precision Krylov loop: FP32 tangent and arithmetic on FP64 vectors
        form_case("jvp", "neohookean", 4, (32, 31, 33), name="neohookean_p4_mixed_jvp", tangent="f32",
                  arithmetic="f32", scatter="colored"),
        # a smoother's operator: BF16 tangent on FP32 vectors
        form_case("jvp", "neohookean", 3, (48, 47, 49), name="neohookean_p3_bf16_jvp", tangent="bf16", vectors="f32"),
        # the Jacobian as a sparse matrix
        form_case("assemble", "neohookean", 2, (14, 12, 13), name="neohookean_p2_assemble", scatter="colored"),
        # one linear system of a mixed-precision Newton step with the multigrid preconditioner
        form_case("mg_solve", "neohookean", 3, (24, 24, 24), name="neohookean_p3_24_mg_solve", tangent="f32",
                  arithmetic="f32"),
        # a bar pulled in two warm-started load steps
        form_case("load_path", "neohookean", 2, (16, 5, 4), name="neohookean_p2_bar_load_path", scatter="colored"),
        # a training step of the network on the vertex grid of the 64^3 mesh
        dict(name="unet_65_train", kind="unet", nx=65, ny=65, nz=65),
    ]


def _elements(rng, lo, hi, flat=2.5):
    """Element counts per direction with a product between about lo and hi, log-uniform, of uneven sides."""
    total = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    side = total ** (1.0 / 3.0)
    a, b = math.exp(rng.uniform(0.0, math.log(flat))), math.exp(rng.uniform(-0.5, 0.5))
    n = [max(1, round(side * a)), max(1, round(side * b / math.sqrt(a))), max(1, round(side / (b * math.sqrt(a))))]
    while n[0] * n[1] * n[2] > hi:
        k = n.index(max(n))
        n[k] -= 1
    rng.shuffle(n)
    return tuple(n)


def draw(rng):
    kind = rng.choice(["residual", "linearize", "linearize", "jvp", "jvp", "jvp", "assemble", "mg_solve", "load_path",
                       "unet"])
    if kind == "unet":
        n = [8 * rng.randint(1, 6) + 1 for _ in range(3)]
        return dict(kind="unet", nx=n[0], ny=n[1], nz=n[2])
    if kind == "mg_solve":
        p = rng.choice([1, 2, 3, 4])
        n = [8 * rng.randint(1, {1: 6, 2: 4, 3: 3, 4: 2}[p]) for _ in range(3)]
        mixed = rng.random() < 0.5
        return form_case(kind, "neohookean", p, n, tangent="f32" if mixed else "f64",
                         arithmetic="f32" if mixed else "f64", scatter=rng.choice(["atomic", "colored"]))
    if kind == "load_path":
        p = rng.choice([1, 2, 3])
        long, wide = {1: (20, 6), 2: (12, 4), 3: (5, 3)}[p]
        return form_case(kind, "neohookean", p, (rng.randint(2, long), rng.randint(2, wide), rng.randint(2, wide)),
                         scatter="colored", perturb=rng.choice([0.0, 0.2]))
    p = rng.choice([1, 2, 3, 4])
    npe = (p + 1) ** 3
    material = rng.choice(["neohookean", "neohookean", "neohookean", "j2", "elastic", "heat", "mass_diffusion"])
    mesh = "cuboid"
    if kind == "assemble":
        n = _elements(rng, 8, 60000 // npe)
    else:
        top = {"residual": 5_000_000, "linearize": 3_500_000, "jvp": 12_000_000}[kind] // npe
        if rng.random() < 0.25:
            mesh, top = "shuffled", min(top, 6000)
        n = _elements(rng, 30, top)
    lin = {"tangent": "f64", "arithmetic": "f64", "vectors": "f64"}
    if kind == "jvp":
        lin["tangent"] = rng.choice(["f64", "f32", "bf16"])
        lin["vectors"] = "f64" if lin["tangent"] == "f64" else rng.choice(["f64", "f32"])
        lin["arithmetic"] = "f64" if lin["tangent"] == "f64" else "f32"
    return form_case(kind, material, p, n, mesh=mesh, perturb=rng.choice([0.0, 0.2]),
                     ordering=rng.choice(["vdim", "vdim", "nodes"]), scatter=rng.choice(["atomic", "colored"]), **lin)


# ---- inputs -----------------------------------------------------------------------------------------------------

def _rule(n):
    """Gauss-Legendre points and weights on [0, 1]."""
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1.0), 0.5 * w


def _nodes_1d(p):
    """Gauss-Lobatto points on [0, 1]."""
    inner = np.polynomial.legendre.Legendre.basis(p).deriv().roots() if p > 1 else np.array([])
    return 0.5 * (np.concatenate([[-1.0], np.sort(inner.real), [1.0]]) + 1.0)


class Grid:
    """The mesh of a case as arrays: vertices, element corners, element nodes (host, numpy)."""

    CORNER_TO_VERTEX = (0, 1, 3, 2, 4, 5, 7, 6)  # lexicographic corner -> place in the hexahedron's vertex list

    def __init__(self, case, seed):
        n = self.n = (case["nx"], case["ny"], case["nz"])
        p = self.p = case["order"]
        h = 1.0 / max(n)
        rng = np.random.RandomState(seed % (2 ** 31))
        vz, vy, vx = np.meshgrid(*[np.arange(k + 1) * h for k in n[::-1]], indexing="ij")
        X = np.stack([vx, vy, vz], axis=-1)
        inside = tuple(slice(1, -1) for _ in range(3))
        if min(n) > 1 and case["perturb"]:
            X[inside] += h * case["perturb"] * rng.uniform(-1.0, 1.0, X[inside].shape)
        self.X, self.h, self.seed, self.rng = X.reshape(-1, 3), h, seed, rng
        ez, ey, ex = (a.ravel() for a in np.meshgrid(*[np.arange(k) for k in n[::-1]], indexing="ij"))
        self.shuffled = case["mesh"] == "shuffled"
        if self.shuffled:
            order = rng.permutation(len(ex))
            ex, ey, ez = ex[order], ey[order], ez[order]
        self.e = (ex, ey, ez)

    def corners(self):
        ex, ey, ez = self.e
        nx, ny = self.n[0] + 1, self.n[1] + 1
        return np.stack([((ez + (c >> 2)) * ny + ey + ((c >> 1) & 1)) * nx + ex + (c & 1) for c in range(8)], axis=1)

    def element_nodes(self):
        """[element][lexicographic node]; shuffled meshes number nodes by first appearance."""
        ex, ey, ez = (a[:, None] * self.p for a in self.e)
        k = np.arange(self.p + 1)
        jz, jy, jx = (a.ravel()[None, :] for a in np.meshgrid(k, k, k, indexing="ij"))
        nx, ny = self.p * self.n[0] + 1, self.p * self.n[1] + 1
        lattice = ((ez + jz) * ny + ey + jy) * nx + ex + jx
        if not self.shuffled:
            return lattice
        _, first, back = np.unique(lattice, return_index=True, return_inverse=True)
        rank = np.empty(len(first), dtype=np.int64)
        rank[np.argsort(first)] = np.arange(len(first))
        return rank[back.reshape(lattice.shape)]

    def nnodes(self):
        return int(np.prod([self.p * k + 1 for k in self.n]))

    def coordinates(self):
        """Node positions of the undisturbed grid on the GPU, [node][3]."""
        g = _nodes_1d(self.p)
        axes = [torch.tensor([(i // self.p + g[i % self.p]) * self.h for i in range(self.p * k + 1)],
                             dtype=torch.float64, device="cuda") for k in self.n]
        z, y, x = torch.meshgrid(*axes[::-1], indexing="ij")
        xyz = torch.stack([x, y, z], dim=-1).reshape(-1, 3)
        if not self.shuffled:
            return xyz
        plain = Grid.element_nodes(_unshuffled(self))
        out = torch.empty_like(xyz)
        out[torch.from_numpy(self.element_nodes().ravel()).cuda()] = xyz[torch.from_numpy(plain.ravel()).cuda()]
        return out

    def build(self):
        if self.shuffled:
            verts = np.empty((len(self.e[0]), 8), dtype=np.int32)
            verts[:, self.CORNER_TO_VERTEX] = self.corners()
            return sx.Mesh.from_arrays(self.X, verts)
        return sx.Mesh.cuboid(*self.n, *[k * self.h for k in self.n])


def _unshuffled(grid):
    """The grid with its shuffled element order and lattice node ids."""
    g = object.__new__(Grid)
    g.__dict__.update(grid.__dict__, shuffled=False)
    return g


def _fields(case, grid, seed):
    """Displacement (temperature) and direction, [node][component] on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    nc = MATERIALS[case["material"]][2]
    xyz = grid.coordinates()

    def noise(amplitude):
        return amplitude * (2.0 * torch.rand(xyz.shape[0], nc, dtype=torch.float64, device="cuda", generator=gen) - 1.0)

    if nc == 1:
        u = torch.sin(math.pi * xyz[:, :1]) + noise(0.5)
    elif case["material"] == "j2":  # simple shear, plastic at most points
        u = torch.stack([0.03 * xyz[:, 2], 0.004 * xyz[:, 0], -0.006 * xyz[:, 2]], dim=1) + noise(2e-3 * grid.h)
    else:  # smooth, with nodal noise that scales with the element size and stays below inverting elements
        # (a linear system is solved at a tenth of it, where the tangent is positive definite)
        base = 0.01 * torch.sin(math.pi * xyz[:, :1])
        u = base * torch.tensor([1.0, 0.5, 0.25], dtype=torch.float64, device="cuda") + noise(0.016 * grid.h)
        if case["kind"] == "mg_solve":
            u = 0.1 * u
    return u, noise(1.0)


def _flat(case, field):
    return (field if case["ordering"] == "vdim" else field.t()).contiguous().reshape(-1)


class Vector:
    """A torch tensor in the place of the framework's DeviceVector: device memory, its length and its type."""

    def __init__(self, tensor):
        self.tensor, self.n = tensor, tensor.numel()
        self.dtype = np.dtype(np.float32 if tensor.dtype == torch.float32 else np.float64)
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


class _Memory:
    """Device memory of the library described for torch."""

    def __init__(self, ptr, n, kind, owner):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (n,), "typestr": kind, "version": 2}
        self.owner = owner


def _tensor(device_vector):
    v = device_vector
    return torch.as_tensor(_Memory(v.ptr.value, v.n, "<f8" if v.dtype == np.float64 else "<f4", v), device="cuda")


def _mesh(case, seed):
    """The mesh; a cuboid's vertices are moved by the library itself, seeded."""
    grid = Grid(dict(case, perturb=0.0 if case["mesh"] == "cuboid" else case["perturb"]), seed)
    mesh = grid.build()
    if case["mesh"] == "cuboid" and case["perturb"]:
        mesh.perturb(seed, case["perturb"])
        grid.X = _perturbed(grid, seed, case["perturb"])
    return grid, mesh


def _mix(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _perturbed(grid, seed, amplitude):
    """The vertices that sx_mesh_perturb gives: a counter-based generator keyed by seed, coordinate and vertex."""
    shape = tuple(k + 1 for k in grid.n[::-1])
    X = grid.X.reshape(shape + (3,)).copy()
    ids = np.arange(int(np.prod(shape)), dtype=np.uint64).reshape(shape)
    inside = tuple(slice(1, -1) for _ in range(3))
    for d in range(3):
        key = _mix(_mix(np.array([seed], dtype=np.uint64)) ^ np.uint64(1000 + d))
        u = (_mix(key ^ ids[inside]) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
        X[inside + (d,)] += grid.h * (-amplitude + 2.0 * amplitude * u)
    return X.reshape(-1, 3)


class State:
    pass


def _form(case, seed):
    s = State()
    s.case = case
    qf, params, nc, _, _ = MATERIALS[case["material"]]
    s.grid, s.mesh = _mesh(case, seed)
    ordering = sx.SX_ORDERING_BYVDIM if case["ordering"] == "vdim" else sx.SX_ORDERING_BYNODES
    s.space = sx.Space(s.mesh, case["order"], nc, ordering)
    s.form = sx.Functional(s.space, [s.space])
    s.form.set_option(capi.SX_OPT_SCATTER,
                      capi.SX_SCATTER_ATOMIC if case["scatter"] == "atomic" else capi.SX_SCATTER_COLORED)
    s.form.set_option(capi.SX_OPT_TANGENT_PRECISION, PRECISION[case["tangent"]])
    if case["vectors"] == "f64":
        s.form.set_option(capi.SX_OPT_JVP_ARITHMETIC, PRECISION[case["arithmetic"]])
    qdata = None
    if case["material"] == "j2":
        qdata = sx.QuadratureData(s.space.ne, (case["order"] + 1) ** 3, J2_STATE)
    s.form.add_domain_integral(qf, params, qdata=qdata)
    u, v = _fields(case, s.grid, seed)
    s.u, s.v = Vector(_flat(case, u)), Vector(_flat(case, v))
    return s


def _end_faces(s):
    return s.space.boundary_dofs(0b11)  # every component on x = 0 and x = max


def prepare(case, seed):
    capi.call("sx_init", torch.cuda.current_device())
    if case["kind"] == "unet":
        return _prepare_unet(case, seed)
    if case["kind"] == "load_path":
        s = _form(case, seed)
        s.ess = _end_faces(s)
        end = s.space.boundary_dofs(0b10, 0b001)
        final = np.zeros(s.space.ndof)
        strain = 0.02 + 0.005 * np.random.RandomState(seed % 2 ** 31).uniform()
        final[end] = strain * s.grid.n[0] * s.grid.h
        s.final = final[s.ess]
        s.x = Vector(torch.zeros(s.space.ndof, dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
        return s
    s = _form(case, seed)
    kind = case["kind"]
    if kind in ("jvp", "assemble", "mg_solve"):
        torch.cuda.synchronize()
        out, s.grad = s.form(0.0, s.u, wrt=0)
    if kind == "mg_solve":  # the system of a Newton step: the residual with the essential rows zeroed
        s.ess = _end_faces(s)
        s.mg = sx.Multigrid(s.space)
        s.v = Vector(_tensor(out).clone())
        s.v.tensor[torch.from_numpy(s.ess.astype(np.int64)).cuda()] = 0.0
    if case["vectors"] == "f32":
        s.v = Vector(s.v.tensor.float())
    s.y = Vector(torch.empty_like(s.v.tensor))
    s.diagonal = Vector(torch.empty(s.space.ndof, dtype=torch.float64, device="cuda"))
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "residual":
        return _tensor(s.form(0.0, s.u))
    if kind == "linearize":
        out, grad = s.form(0.0, s.u, wrt=0)
        grad.diagonal(s.diagonal)
        grad.mult(s.v, s.y)
        return {"residual": _tensor(out), "diagonal": s.diagonal.tensor, "jv": s.y.tensor}
    if kind == "jvp":
        s.grad.mult(s.v, s.y)
        return s.y.tensor
    if kind == "assemble":
        A = s.grad.assemble()
        A.mult(s.v, s.y)
        val = ctypes.c_void_p()
        capi.call("sx_csr_arrays", A.h, None, None, ctypes.byref(val))
        values = _Memory(val.value, A.nnz, "<f8", A)
        return {"values": torch.as_tensor(values, device="cuda"), "product": s.y.tensor}
    if kind == "mg_solve":
        s.grad.mg_cg(s.mg, s.ess, s.v, s.y, rel_tol=1e-8)
        return s.y.tensor
    if kind == "load_path":
        s.x.tensor.zero_()
        torch.cuda.current_stream().synchronize()  # the solver works on a stream of its own
        sx.quasistatic_solve(s.form, s.x, s.ess, s.final, 2, rel_tol=1e-8, lin_rel_tol=1e-6)
        return s.x.tensor
    loss = s.net.backward(s.x, s.t)
    grads = s.net.grads()
    s.net.adam(1e-4)
    return {"loss": loss, "gradients": grads}


# ---- what a pass cannot do without ------------------------------------------------------------------------------

def work(case):
    if case["kind"] == "unet":
        n = [(case["nx"], case["ny"], case["nz"])]
        for _ in range(3):
            n.append(tuple((k - 1) // 2 + 1 for k in n[-1]))
        vox = [a * b * c for a, b, c in n]
        level = [0, 0, 1, 1, 2, 2, 3, 3, 2, 1, 0, 0]
        flops = sum(3 * 2 * 27 * (a + b) * c * vox[lv] for (a, b, c), lv in zip(sx.UNet.LAYERS, level))
        # input and target, the master weights, both Adam moments and the gradients
        return {"bytes": 24 * vox[0] + 32 * sum(27 * (a + b) * c + c for a, b, c in sx.UNet.LAYERS), "flops": flops}
    p = case["order"]
    _, _, nc, entries, inputs = MATERIALS[case["material"]]
    ne = case["nx"] * case["ny"] * case["nz"]
    N = p + 1
    nqp = npe = N ** 3
    nodes = (p * case["nx"] + 1) * (p * case["ny"] + 1) * (p * case["nz"] + 1)
    ndof = nodes * nc
    maps, geometry = 4 * ne * npe, 24 * (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
    sv, sd = BYTES[case["vectors"]], BYTES[case["tangent"]]
    tangent = sd * entries * nqp * ne
    contract = 2 * 2 * 8 * nc * N * nqp * ne  # interpolation and integration by sum factorization
    state = 80 * nqp * ne if case["material"] == "j2" else 0
    point = {"heat": 40, "mass_diffusion": 150, "elastic": 130, "neohookean": 320, "j2": 450}[case["material"]] * nqp * ne
    jvp = {"bytes": 2 * sv * ndof + tangent + maps, "flops": contract + 2 * inputs ** 2 * nqp * ne}
    residual = {"bytes": 16 * ndof + geometry + maps + state, "flops": contract + point}
    if case["kind"] == "residual":
        return residual
    if case["kind"] == "jvp":
        return jvp
    diagonal = {"bytes": tangent * 6 * nc // entries + 8 * ndof + maps, "flops": 2 * 6 * 3 * nc * N * nqp * ne}
    linearize = {"bytes": residual["bytes"] + tangent, "flops": residual["flops"] + 5 * entries * nqp * ne}
    if case["kind"] == "linearize":
        parts = [linearize, diagonal, jvp]
        return {k: sum(q[k] for q in parts) for k in ("bytes", "flops")}
    if case["kind"] == "assemble":
        # the element blocks column by column through the sum factorization; values and columns written, read once
        nnz = nc * nc * ((2 * p + 1) * p ** 2 * ne if p > 1 else 27 * ne) * 4
        return {"bytes": tangent + maps + 20 * nnz, "flops": npe * nc * (contract // 2 + 2 * inputs ** 2 * nqp * ne) // 8}
    if case["kind"] == "mg_solve":  # about 50 iterations of five operator applications and the streams between them
        return {"bytes": 250 * jvp["bytes"] + 50 * 40 * 8 * ndof, "flops": 250 * jvp["flops"]}
    # about six linear solves of 1000 Jacobi-CG iterations
    return {"bytes": 6000 * (jvp["bytes"] + 112 * ndof), "flops": 6000 * jvp["flops"]}


def tolerance(case):
    """About four times the difference between two orders of summation (or between these results and exact())."""
    if case["kind"] == "unet":  # BF16 activations: a product summed in another order changes a rounding
        return {"rel": 1e-2}
    if case["kind"] == "mg_solve":  # the solve stops at 1e-8 in the preconditioned norm, an iteration sooner or later
        return {"rel": 4e-7}
    if case["kind"] == "load_path":  # an iteration sooner or later in a linear solve that Newton corrects
        return {"rel": 1e-9}
    if case["kind"] == "jvp" and case["tangent"] != "f64":  # both tangents are the FP64 one, rounded once
        return {"rel": 1e-6}
    return {"rel": 2e-13}


# ---- the same results from plain torch in 64 bits ---------------------------------------------------------------

def _tables(p):
    """B[q][i], G[q][i]: the Lobatto-Lagrange basis and its derivative at the Gauss points, and the weights."""
    x, q_w = _nodes_1d(p), _rule(p + 1)
    q, w = q_w
    n = p + 1
    B, G = np.ones((n, n)), np.zeros((n, n))
    for i in range(n):
        others = [j for j in range(n) if j != i]
        for a in range(n):
            B[a, i] = np.prod([(q[a] - x[j]) / (x[i] - x[j]) for j in others])
            G[a, i] = sum(np.prod([(q[a] - x[j]) / (x[i] - x[j]) for j in others if j != k]) / (x[i] - x[k])
                          for k in others)
    dev = dict(dtype=torch.float64, device="cuda")
    return torch.tensor(B, **dev), torch.tensor(G, **dev), torch.tensor(q, **dev), torch.tensor(w, **dev)


def _inverse3(A):
    """Inverse and determinant of [..., 3, 3] by cofactors."""
    a, b, c = A[..., 0, :], A[..., 1, :], A[..., 2, :]
    rows = torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)], dim=-1)
    det = (a * rows[..., :, 0]).sum(-1)
    return rows / det[..., None, None], det


def _flux(material, params):
    """(value [.., c], grad [.., c, 3]) -> (source, flux) at the points, in physical space."""
    eye = torch.eye(3, dtype=torch.float64, device="cuda")

    def heat(v, g):
        return torch.zeros_like(v) - params[1], params[0] * g

    def mass_diffusion(v, g):
        return params[0] * v, params[1] * g

    def elastic(v, g):
        tr = g.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]
        return torch.zeros_like(v), params[1] * (g + g.transpose(-1, -2)) + params[0] * tr * eye

    def neohookean(v, H):
        K, G = params[1], params[2]
        Hd, Ht = H, H.transpose(-1, -2)
        tr = Hd.diagonal(dim1=-2, dim2=-1).sum(-1)
        sq = (Hd * Ht).sum((-1, -2))
        det = (Hd[..., 0, :] * torch.linalg.cross(Hd[..., 1, :], Hd[..., 2, :])).sum(-1)
        jm1 = tr + 0.5 * (tr * tr - sq) + det
        tau = (K - 2.0 * G / 3.0) * torch.log1p(jm1)[..., None, None] * eye
        tau = tau + G * ((Hd[..., :, None, :] * Hd[..., None, :, :]).sum(-1) + Hd + Ht)
        Fi, _ = _inverse3(Hd + eye)
        return torch.zeros_like(v), (tau[..., :, None, :] * Fi[..., None, :, :]).sum(-1)

    def j2(v, H):
        E, nu, sy, Hi, Hk = params[:5]
        K, G = E / (3.0 * (1.0 - 2.0 * nu)), 0.5 * E / (1.0 + nu)
        ep = torch.tensor(J2_STATE[:9], dtype=torch.float64, device="cuda").reshape(3, 3)
        el = 0.5 * (H + H.transpose(-1, -2)) - ep
        tr = el.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]
        s = 2.0 * G * (el - tr / 3.0 * eye)
        eta = s - (2.0 / 3.0) * Hk * ep
        q = math.sqrt(1.5) * (eta * eta).sum((-1, -2)).sqrt()
        over = q - (sy + Hi * J2_STATE[9])
        delta = torch.where(over > 1e-10 * sy, over / (3.0 * G + Hk + Hi), torch.zeros_like(over))
        s = s - (3.0 * G * delta / q)[..., None, None] * eta + K * tr * eye
        Fi, det = _inverse3(H + eye)
        return torch.zeros_like(v), (s[..., :, None, :] * Fi[..., None, :, :]).sum(-1) * det[..., None, None]

    return {"heat": heat, "mass_diffusion": mass_diffusion, "elastic": elastic, "neohookean": neohookean, "j2": j2}[material]


class Reference:
    """The weak form of a case by dense torch operations, chunks of elements at a time."""

    def __init__(self, case, seed):
        _, self.params, self.nc, _, _ = MATERIALS[case["material"]]
        self.case, self.N = case, case["order"] + 1
        self.flux = _flux(case["material"], self.params)
        grid = Grid(dict(case, perturb=0.0 if case["mesh"] == "cuboid" else case["perturb"]), seed)
        if case["mesh"] == "cuboid" and case["perturb"]:
            grid.X = _perturbed(grid, seed, case["perturb"])
        self.grid, self.nn = grid, grid.nnodes()
        self.emap = torch.from_numpy(grid.element_nodes()).cuda()
        self.corners = torch.from_numpy(grid.X[grid.corners()]).cuda()
        self.B, self.G, self.q, self.w = _tables(case["order"])
        self.u, self.v = _fields(case, grid, seed)
        self.chunk = max(1, 400_000 // self.N ** 3)

    def chunks(self):
        for a in range(0, len(self.emap), self.chunk):
            yield slice(a, min(a + self.chunk, len(self.emap)))

    def geometry(self, k):
        """Inverse Jacobian and weighted determinant at the points of the elements k, points (z, y, x)."""
        x = self.q
        n1 = torch.stack([1.0 - x, x])
        d1 = torch.stack([-torch.ones_like(x), torch.ones_like(x)])
        X = self.corners[k].reshape(-1, 2, 2, 2, 3)  # corner (z, y, x)
        J = torch.stack([torch.einsum("ecbai,cz,by,ax->ezyxi", X, *t) for t in
                         ((n1, n1, d1), (n1, d1, n1), (d1, n1, n1))], dim=-1)
        Ji, det = _inverse3(J)
        w = self.w[:, None, None] * self.w[:, None] * self.w
        return Ji, det * w

    def _along(self, T, axes):
        for axis, table in axes:
            T = torch.tensordot(T, table, dims=([axis], [1])).movedim(-1, axis)
        return T

    def interpolate(self, k, field, Ji):
        """Values and physical gradients of a nodal field [node][c] at the points."""
        U = field[self.emap[k]].reshape(-1, self.N, self.N, self.N, self.nc)
        B, G = self.B, self.G
        val = self._along(U, ((1, B), (2, B), (3, B)))
        gp = torch.stack([self._along(U, t) for t in (((1, B), (2, B), (3, G)), ((1, B), (2, G), (3, B)),
                                                      ((1, G), (2, B), (3, B)))], dim=-1)
        return val, self.to_physical(gp, Ji)

    @staticmethod
    def to_physical(gp, Ji):
        return (gp[..., :, :, None] * Ji[..., None, :, :]).sum(-2)

    def integrate(self, k, source, flux, Ji, wdet, out):
        B, G = self.B.t(), self.G.t()
        fp = (flux[..., :, None, :] * Ji[..., None, :, :]).sum(-1) * wdet[..., None, None]
        r = self._along(source * wdet[..., None], ((1, B), (2, B), (3, B)))
        for d, t in enumerate((((1, B), (2, B), (3, G)), ((1, B), (2, G), (3, B)), ((1, G), (2, B), (3, B)))):
            r = r + self._along(fp[..., d], t)
        out.index_add_(0, self.emap[k].reshape(-1), r.reshape(-1, self.nc))

    def residual(self, with_jv=True):
        r, jv = torch.zeros_like(self.u), torch.zeros_like(self.u)
        for k in self.chunks():
            Ji, wdet = self.geometry(k)
            at = self.interpolate(k, self.u, Ji)
            if with_jv:
                (s, f), (ds, df) = torch.func.jvp(self.flux, at, self.interpolate(k, self.v, Ji))
                self.integrate(k, ds, df, Ji, wdet, jv)
            else:
                s, f = self.flux(*at)
            self.integrate(k, s, f, Ji, wdet, r)
        return r, jv

    def tangent(self, k):
        """D[e, q, (value, parent gradient) of each component out, the same in] with the weights, 4 nc each way."""
        Ji, wdet = self.geometry(k)
        val, g = self.interpolate(k, self.u, Ji)
        columns = []
        for c in range(self.nc):
            for a in range(4):
                dv, dg = torch.zeros_like(val), torch.zeros_like(g)
                if a == 0:
                    dv[..., c] = 1.0
                else:
                    dg[..., c, :] = Ji[..., a - 1, :]
                _, (ds, df) = torch.func.jvp(self.flux, (val, g), (dv, dg))
                fp = (df[..., :, None, :] * Ji[..., None, :, :]).sum(-1)
                columns.append(torch.cat([ds[..., None], fp], dim=-1) * wdet[..., None, None])
        D = torch.stack(columns, dim=-1)  # [e, z, y, x, c, 4, 4 nc]
        ne = D.shape[0]
        return D.reshape(ne, self.N ** 3, self.nc, 4, self.nc, 4)

    def shape_functions(self):
        """[q, node, 4]: value and parent gradient of every basis function at every point."""
        B, G = self.B, self.G
        parts = [torch.einsum("ck,bj,ai->cbakji", *t).reshape(self.N ** 3, self.N ** 3) for t in
                 ((B, B, B), (B, B, G), (B, G, B), (G, B, B))]
        return torch.stack(parts, dim=-1)

    def diagonal(self):
        phi, out = self.shape_functions(), torch.zeros_like(self.u)
        pair = (phi[..., :, None] * phi[..., None, :]).permute(0, 2, 3, 1).reshape(-1, self.N ** 3)
        for k in self.chunks():
            D = self.tangent(k)
            block = torch.stack([D[:, :, c, :, c, :] for c in range(self.nc)], dim=1)  # [e, c, q, 4, 4]
            d = block.reshape(block.shape[0] * self.nc, -1) @ pair
            out.index_add_(0, self.emap[k].reshape(-1),
                           d.reshape(-1, self.nc, self.N ** 3).transpose(1, 2).reshape(-1, self.nc))
        return out

    def dof(self, node, c):
        return node * self.nc + c if self.case["ordering"] == "vdim" else c * self.nn + node

    def element_matrices(self, k):
        phi, D = self.shape_functions(), self.tangent(k)
        ne, nq, M, nd = D.shape[0], self.N ** 3, 4 * self.nc, self.nc * self.N ** 3
        # T[q, (c, a), (c, j)] = phi of node j, input a
        T = torch.zeros(nq, self.nc, 4, self.nc, nq, dtype=torch.float64, device="cuda")
        for c in range(self.nc):
            T[:, c, :, c, :] = phi.permute(0, 2, 1)
        T = T.reshape(nq * M, nd)
        right = torch.matmul(D.reshape(ne, nq, M, M), T.reshape(nq, M, nd)).reshape(ne, nq * M, nd)
        return torch.matmul(T.t().contiguous(), right)

    def matrix(self):
        """The assembled matrix as sorted COO (rows, columns, values)."""
        where, values = [], []
        ndof = self.nn * self.nc
        c = torch.arange(self.nc, device="cuda")[:, None]
        for a in range(0, len(self.emap), 64):
            k = slice(a, min(a + 64, len(self.emap)))
            dofs = self.dof(self.emap[k][:, None, :], c).reshape(k.stop - k.start, -1)
            where.append((dofs[:, :, None] * ndof + dofs[:, None, :]).reshape(-1))
            values.append(self.element_matrices(k).reshape(-1))
        key, back = torch.unique(torch.cat(where), return_inverse=True)
        val = torch.zeros(len(key), dtype=torch.float64, device="cuda").index_add_(0, back, torch.cat(values))
        return key // ndof, key % ndof, val


def exact(case, seed):
    kind = case["kind"]
    if kind == "unet":
        return _exact_unet(case, seed)
    if kind in ("mg_solve", "load_path"):
        return None
    ref = Reference(case, seed)
    if kind == "residual":
        return _flat(case, ref.residual(False)[0])
    if kind == "linearize":
        r, jv = ref.residual()
        return {"residual": _flat(case, r), "diagonal": _flat(case, ref.diagonal()), "jv": _flat(case, jv)}
    if kind == "jvp":
        if case["vectors"] == "f32":
            ref.v = ref.v.float().double()
        return _flat(case, ref.residual()[1])
    row, col, val = ref.matrix()
    x = _flat(case, ref.v)
    return {"values": val, "product": torch.zeros_like(x).index_add_(0, row, val * x[col])}


# ---- the network ------------------------------------------------------------------------------------------------

def _unet_data(case, seed):
    """Parameters (normal, variance 2 / fan-in), a restricted residual and a smoother correction on the grid."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    params = []
    for a, b, c in sx.UNet.LAYERS:
        params.append(torch.randn(27 * (a + b) * c, device="cuda", generator=gen) * math.sqrt(2.0 / (27 * (a + b))))
        params.append(0.05 * torch.randn(c, device="cuda", generator=gen))
    shape = (case["nz"], case["ny"], case["nx"], 3)
    x = torch.randn(shape, device="cuda", generator=gen)
    z, y, w = (torch.linspace(0.0, 1.0, k, device="cuda") for k in shape[:3])
    smooth = torch.sin(math.pi * z)[:, None, None] * torch.sin(math.pi * y)[:, None] * torch.sin(2 * math.pi * w)
    t = smooth[..., None] * torch.tensor([1.0, -0.5, 0.25], device="cuda") + 0.1 * torch.randn(shape, device="cuda",
                                                                                               generator=gen)
    return torch.cat(params), x.contiguous(), t.contiguous()


def _prepare_unet(case, seed):
    s = State()
    s.case = case
    params, x, t = _unet_data(case, seed)
    s.net = sx.UNet(case["nx"], case["ny"], case["nz"])
    s.net.set_params(params.cpu().numpy())
    s.x = sx.DeviceVector.from_numpy(x.cpu().numpy(), dtype=np.float32)
    s.t = sx.DeviceVector.from_numpy(t.cpu().numpy(), dtype=np.float32)
    torch.cuda.synchronize()
    return s


def _exact_unet(case, seed):
    flat, x, t = _unet_data(case, seed)
    leaf = flat.double().requires_grad_(True)
    weights, at = [], 0
    for a, b, c in sx.UNet.LAYERS:
        w = leaf[at:at + 27 * (a + b) * c].reshape(27, a + b, c)
        w = w + (w.float().bfloat16().double() - w).detach()  # BF16 weights, gradients to the masters
        weights.append((w, leaf[at + w.numel():at + w.numel() + c]))
        at += w.numel() + c

    def conv(k, x, stride=1):
        w, bias = weights[k]
        padded = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        n = x.shape
        y = bias.clone()
        for tap in range(27):
            i, j, m = tap // 9, (tap // 3) % 3, tap % 3
            y = y + padded[i:i + n[0]:stride, j:j + n[1]:stride, m:m + n[2]:stride] @ w[tap]
        return y

    def prolong(x):
        for axis in range(3):
            x = x.movedim(axis, 0)
            mid = 0.5 * (x[:-1] + x[1:])
            x = torch.cat([torch.stack([x[:-1], mid], dim=1).flatten(0, 1), x[-1:]]).movedim(0, axis)
        return x

    relu = torch.relu
    a0 = relu(conv(0, x.bfloat16().double()))
    b0 = relu(conv(1, a0))
    b1 = relu(conv(3, relu(conv(2, b0, 2))))
    b2 = relu(conv(5, relu(conv(4, b1, 2))))
    b3 = relu(conv(7, relu(conv(6, b2, 2))))
    c2 = relu(conv(8, torch.cat([prolong(b3), b2], dim=-1)))
    c1 = relu(conv(9, torch.cat([prolong(c2), b1], dim=-1)))
    c0 = relu(conv(10, torch.cat([prolong(c1), b0], dim=-1)))
    loss = (conv(11, c0) - t.double()).square().sum() / t.double().square().sum()
    loss.backward()
    return {"loss": float(loss.detach()), "gradients": leaf.grad.detach()}
