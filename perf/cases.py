"""The work that programs have this framework do, as cases that can be timed and compared.

A case is a dict of plain values.  "kind" names the call:

- "newton": one solver.solver(...) call on host data, the framework's main entry: assembly, Newton
  and the (Jacobi- or network-) preconditioned Krylov solve.  "model": Poisson with a source,
  variable-coefficient Poisson, the plane-strain Neo-Hooke panel under a traction (2 DOFs per
  node), or the Neo-Hooke cube of Hex8 bricks (3 DOFs per node).  "precision": FP64 or mixed.
- "assemble": residual and reduced tangent on device arrays through the C ABI, for a program that
  runs its own nonlinear solver.
- "pairs": learned.solver_pairs, the plain solve (matrix in canonical CSR order, on the device)
  that makes a training pair.
- "train": one training step of the network (forward, loss, backward, Adam).
- "sensitivity": reverse-mode sensitivities of a Q2 'user element' solution
  (implicit_diff.root_vjp: tangent, adjoint solve, parameter derivatives).

Sizes are elements per direction.  Meshes, plans and models are made once per size and kept, as a
program that solves many times on one mesh keeps them; what a seed changes is what changes from call
to call: boundary values, fields, loads, material, displacements, weights, right-hand sides.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from autopdex_amd import _native, backend, geometry, implicit_diff, learned, mesher, models, seeder, solver, spaces
from autopdex_amd import utility

PANEL = ((0.0, 0.0), (48.0, 44.0), (48.0, 60.0), (0.0, 44.0))
CUBE = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))
SOURCE = (20.0, 10.0, 1.0, 0.5)  # amplitude, frequency and centre of the Poisson source


def listed():
    return [
        # the smallest call: a quick-start-sized Poisson problem, DOFs in a dict; launches and host work
        dict(name="newton_poisson_16", kind="newton", model="poisson", nx=16, ny=16, nz=0, skew=False,
             precision="fp64", precond="jacobi"),
        # an ordinary 2D solve to solver accuracy (40 k DOFs)
        dict(name="newton_poisson_200", kind="newton", model="poisson", nx=200, ny=200, nz=0, skew=False,
             precision="fp64", precond="jacobi"),
        # a new coefficient field on a general quadrilateral, odd sizes, mixed precision
        dict(name="newton_vark_1023x771", kind="newton", model="vark", nx=1023, ny=771, nz=0, skew=True,
             precision="mixed", precond="jacobi"),
        # the largest: the 4.2 M DOF Poisson problem with the plain FP64 method
        dict(name="newton_poisson_2048", kind="newton", model="poisson", nx=2048, ny=2048, nz=0, skew=False,
             precision="fp64", precond="jacobi"),
        # the same problem family with the network preconditioner and the FP32 matrix
        dict(name="newton_learned_1024", kind="newton", model="poisson", nx=1024, ny=1024, nz=0, skew=False,
             precision="mixed", precond="learned"),
        # a load step of the nearly incompressible panel: nonlinear, many Krylov iterations on a small system
        dict(name="newton_panel_64x48", kind="newton", model="panel", nx=64, ny=48, nz=0, skew=False,
             precision="fp64", precond="jacobi"),
        # a load step of the 3D cube with the FP32 tangent
        dict(name="newton_cube_20", kind="newton", model="cube", nx=20, ny=19, nz=21, skew=False,
             precision="mixed", precond="jacobi"),
        # assembly of the 3D configuration at full size (823,875 DOFs)
        dict(name="assemble_cube_64", kind="assemble", model="cube", nx=64, ny=64, nz=64, skew=False),
        # assembly of the plane-strain configuration at full size (526,338 DOFs)
        dict(name="assemble_panel_512", kind="assemble", model="panel", nx=512, ny=512, nz=0, skew=False),
        # a training pair at a size that the network is trained on
        dict(name="pairs_512x384", kind="pairs", model="poisson", nx=512, ny=384, nz=0, skew=False),
        # a training step with the batch that learned.fit uses
        dict(name="train_512", kind="train", model="poisson", nx=512, ny=512, nz=0, skew=False, batch=4),
        # sensitivities of a Cook's-membrane-like Q2 solution with respect to E and nu
        dict(name="sensitivity_q2_16x12", kind="sensitivity", model="q2", nx=16, ny=12, nz=0, skew=False),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("newton", "newton", "newton", "newton", "assemble", "assemble", "pairs", "train", "sensitivity"))
    c = dict(kind=kind, nz=0, skew=False)
    if kind == "newton":
        c["model"] = rng.choice(("poisson", "vark", "panel", "cube"))
        c["precision"] = rng.choice(("fp64", "mixed"))
        c["precond"] = "jacobi"
        if c["model"] in ("poisson", "vark"):
            c["nx"], c["ny"] = _log_int(rng, 6, 1500), _log_int(rng, 6, 1500)
            c["skew"] = rng.random() < 0.5
            if c["model"] == "poisson" and rng.random() < 0.3:
                c.update(precond="learned", skew=False, nx=_log_int(rng, 64, 1200))
                c["ny"] = int(c["nx"] * rng.uniform(0.7, 1.3))
        elif c["model"] == "panel":
            c["nx"], c["ny"] = _log_int(rng, 6, 72), _log_int(rng, 6, 56)
        else:
            c["nx"], c["ny"], c["nz"] = (_log_int(rng, 3, 24) for _ in range(3))
    elif kind == "assemble":
        c["model"] = rng.choice(("vark", "panel", "cube", "q2"))
        if c["model"] == "cube":
            c["nx"], c["ny"], c["nz"] = (_log_int(rng, 5, 62) for _ in range(3))
        else:
            top = {"vark": 1800, "panel": 600, "q2": 300}[c["model"]]
            c["nx"], c["ny"] = _log_int(rng, 12, top), _log_int(rng, 12, top)
            c["skew"] = c["model"] == "vark" and rng.random() < 0.5
    elif kind == "pairs":
        c["model"] = "poisson"
        c["nx"], c["ny"] = _log_int(rng, 12, 700), _log_int(rng, 12, 700)
    elif kind == "train":
        c["model"] = "poisson"
        c["nx"] = _log_int(rng, 48, 600)
        c["ny"] = int(c["nx"] * rng.uniform(0.7, 1.3))
        c["batch"] = rng.choice((1, 2, 4))
    else:
        c["model"] = "q2"
        c["nx"], c["ny"] = _log_int(rng, 4, 20), _log_int(rng, 4, 16)
    return c


# ---- meshes and settings ------------------------------------------------------------------------

def _q2_mesh(nx, ny):
    """A tapered membrane of nx x ny 9-node quads and the 3-node lines of its right edge."""
    coords, _ = mesher.structured_mesh((2 * nx, 2 * ny), PANEL, "quad")
    m = 2 * ny + 1
    i, j = (a.ravel() for a in np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij"))
    at = lambda di, dj: (2 * i + di) * m + 2 * j + dj  # noqa: E731
    offsets = ((0, 0), (2, 0), (2, 2), (0, 2), (1, 0), (2, 1), (1, 2), (0, 1), (1, 1))
    elems = np.stack([at(*o) for o in offsets], axis=1).astype(np.int64)
    k = 2 * nx * m + 2 * np.arange(ny)
    return coords, elems, np.stack([k, k + 2, k + 1], axis=1).astype(np.int64)


@functools.lru_cache(maxsize=3)
def _mesh(model, nx, ny, nz, skew):
    """(coords, element sets, Dirichlet mask, static settings): what a program keeps per mesh."""
    static = {"solution structure": ("nodal imposition",), "solver type": "newton", "solver backend": "hip",
              "solver": "cg", "type of preconditioner": "jacobi", "verbose": -1}
    if model in ("poisson", "vark"):
        verts = ((0.0, 0.0), (2.0, 0.0), (2.0, 0.7), (0.0, 1.0)) if skew else (
            (0.0, 0.0), (1.0, 0.0), (1.0, ny / nx), (0.0, ny / nx))
        coords, elems = mesher.structured_mesh((nx, ny), verts, "quad")
        mask = geometry.in_sdfs(coords, lambda x: geometry.psdf_polygon(x, [list(v) for v in verts]))
        integrand = (models.poisson_source_integrand() if model == "poisson"
                     else models.poisson_variable_coefficient_integrand("log coefficient", "source"))
        pot = models.mixed_reference_domain_potential(integrand, {"u": spaces.fem_iso_line_quad_brick},
                                                      *seeder.gauss_legendre_nd(2, 2), "u")
        sets, mods, mode = (elems,), (pot,), "user potential"
    elif model == "panel":
        coords, elems = mesher.structured_mesh((nx, ny), PANEL, "quad")
        mask = utility.dof_select(geometry.in_planes(coords, [0, 0], [1, 0]), [True, True])
        pot = models.mixed_reference_domain_potential(
            models.hyperelastic_integrand(models.neo_hooke, "lam", "mu"), {"u": spaces.fem_iso_line_quad_brick},
            *seeder.gauss_legendre_nd(2, 2), "u")
        trac = models.line_traction_potential(np.array([0.0, 1.0 / 16.0]), "load multiplier")
        sets, mods, mode = (elems, mesher.boundary_lines((nx, ny), "right")), (pot, trac), "user potential"
    elif model == "cube":
        coords, elems = mesher.structured_mesh((nx, ny, nz), CUBE, "brick")
        left, right = (geometry.in_planes(coords, [x, 0, 0], [1, 0, 0]) for x in (0, 1))
        mask = utility.dof_select(left, [True, True, True]) | utility.dof_select(right, [True, False, False])
        pot = models.mixed_reference_domain_potential(
            models.hyperelastic_integrand(models.neo_hooke, "lam", "mu"), {"u": spaces.fem_iso_line_quad_brick},
            *seeder.gauss_legendre_nd(3, 2), "u")
        sets, mods, mode = (elems,), (pot,), "user potential"
    else:
        coords, elems, lines = _q2_mesh(nx, ny)
        mask = utility.dof_select(geometry.in_planes(coords, [0, 0], [1, 0]), [True, True])
        weak = models.hyperelastic_steady_state_weak(models.neo_hooke, lambda x, s: s["youngs modulus"],
                                                     lambda x, s: s["poisson ratio"], "plain strain")
        elem = models.isoparametric_domain_element_galerkin(weak, spaces.fem_iso_line_quad_brick,
                                                            *seeder.gauss_legendre_nd(dimension=2, order=4))
        load = models.neumann_weak(lambda x, s: np.asarray([0.0, s["load multiplier"]]))
        surf = models.isoparametric_surface_element_galerkin(load, spaces.fem_iso_line_quad_brick,
                                                             *seeder.gauss_legendre_nd(dimension=1, order=4),
                                                             tangent_contributions=False)
        sets, mods, mode = (elems, lines), (elem, surf), "user element"
    static["model"], static["assembling mode"] = mods, tuple(mode for _ in mods)
    return coords, sets, mask, static


def _waves(coords, rng, waves=6, most=5.0):
    """A smooth random field (zero mean, about unit size) at the given points."""
    f = np.zeros(coords.shape[0])
    size = np.ptp(coords, axis=0).max()
    for _ in range(waves):
        f += rng.standard_normal() * np.cos(coords @ (rng.uniform(-most, most, coords.shape[1]) / size)
                                            + rng.uniform(0, 2 * math.pi))
    return f * math.sqrt(2.0 / waves)


def _inputs(c, seed):
    """(dofs, settings, static settings) of one call."""
    coords, sets, mask, static = _mesh(c["model"], c["nx"], c["ny"], c["nz"], c["skew"])
    rng = np.random.default_rng(seed)
    dofs, values = np.zeros(mask.shape), np.zeros(mask.shape)
    s = {"connectivity": sets, "dirichlet dofs": mask, "node coordinates": coords, "dirichlet conditions": values}
    if c["model"] in ("poisson", "vark"):
        values[mask] = 0.1 * _waves(coords[mask], rng)
        if c["model"] == "vark":
            s["log coefficient"], s["source"] = _waves(coords, rng, 8, 40.0), rng.standard_normal(mask.size)
    elif c["model"] == "panel":
        s.update({"lam": 40.0 * rng.uniform(0.9, 1.1), "mu": 0.4 * rng.uniform(0.9, 1.1),
                  "load multiplier": 0.1 * rng.uniform(0.8, 1.2)})
    elif c["model"] == "cube":
        s.update({"lam": 10.0 * rng.uniform(0.9, 1.1), "mu": rng.uniform(0.9, 1.1)})
        pull = 0.02 * rng.uniform(0.8, 1.2)
        values[:, 0] = np.where(mask[:, 0], pull * coords[:, 0], 0.0)
        dofs[:, 0] = pull * coords[:, 0]  # the last load step's solution extended linearly
    else:
        s.update({"youngs modulus": 100.0 * rng.uniform(0.9, 1.1), "poisson ratio": 0.3 * rng.uniform(0.9, 1.1),
                  "load multiplier": 4.0 * rng.uniform(0.8, 1.2)})
    if c["model"] == "poisson" and c["nx"] <= 16 and c["ny"] <= 16:  # the quick-start form: DOFs in a dict
        for k in ("dirichlet dofs", "node coordinates", "dirichlet conditions"):
            s[k] = {"u": s[k]}
        s["connectivity"], dofs = _dict_sets(c["model"], c["nx"], c["ny"], c["nz"], c["skew"]), {"u": dofs}
    static = dict(static)
    if c["kind"] == "newton":
        nonlinear = c["model"] in ("panel", "cube")
        static.update({"hip precision": c["precision"], "type of preconditioner": c["precond"],
                       "linear tolerance": 1e-12 if c["precision"] == "fp64" else 1e-6})
        if not nonlinear:
            static.update({"newton tolerance mode": "relative", "linear forcing": True})
        if c["precond"] == "learned":
            static["reliable delta"] = 1e-2
    return dofs, s, static


@functools.lru_cache(maxsize=3)
def _dict_sets(*key):
    return tuple({"u": e} for e in _mesh(*key)[1])


def _displacement(c, coords, seed):
    """A smooth displacement of a few percent strain, with a little of every wave length."""
    rng = np.random.default_rng(seed)
    size, d = np.ptp(coords, axis=0).max(), coords.shape[1]
    u = np.stack([0.004 * size * _waves(coords, rng) for _ in range(d)], axis=1)
    return u + 0.01 * size / max(c["nx"], c["ny"], c["nz"]) * rng.standard_normal(u.shape)


# ---- the network --------------------------------------------------------------------------------

def _levels(h, w):
    n = 1
    while n < 12 and min((h + 1) // 2, (w + 1) // 2) >= 3:
        h, w, n = (h + 1) // 2, (w + 1) // 2, n + 1
    return n


def _channels(levels):
    return ((16, 32) + (64,) * 10)[:levels]


def _layers(levels):
    """(role, level, input channels, output channels) in the order of the parameter vector."""
    ch = _channels(levels)
    out = [("in", 0, 1, ch[0])]
    for l in range(levels - 1):
        out += [("e", l, ch[l], ch[l]), ("down", l, ch[l], ch[l + 1])]
    out.append(("b", levels - 1, ch[-1], ch[-1]))
    for l in range(levels - 2, -1, -1):
        out += [("up", l, ch[l + 1], ch[l]), ("d", l, ch[l], ch[l])]
    return out + [("out", 0, ch[0], 1)]


def _layout(levels):
    """Each layer with the place and padded shape of its weights in the parameter vector."""
    off = 0
    for role, l, ci, co in _layers(levels):
        cop, wk = (co + 15) // 16 * 16, (9 * ci if ci >= 16 else (9 * ci + 15) // 16 * 16)
        yield role, l, ci, co, cop, wk, off
        off += cop * wk + co
    yield "end", 0, 0, 0, 0, 0, off


def _theta(levels, fill):
    """The parameter vector with fill(role, level, ci, co) -> (co, 9, ci) weights and no biases."""
    layout = list(_layout(levels))
    theta = np.zeros(layout[-1][-1], dtype=np.float32)
    for role, l, ci, co, cop, wk, off in layout[:-1]:
        w = np.zeros((cop, wk), dtype=np.float32)
        w[:co, :9 * ci] = fill(role, l, ci, co).reshape(co, 9 * ci)
        theta[off:off + cop * wk] = w.ravel()
    return theta


def _starting_weights(levels, seed):
    """He-normal weights with small coarse branches: what training starts from."""
    rng = np.random.default_rng(seed)
    scale = {"up": 0.05, "out": 0.1}

    def fill(role, l, ci, co):
        return rng.standard_normal((co, 9, ci)) * scale.get(role, 1.0) / math.sqrt(9 * ci)

    return _theta(levels, fill)


def _multilevel_weights(levels, seed):
    """Weights whose network is an additive multilevel preconditioner: every layer acts at the
    centre tap, the channels carry the residual along random isometries, each coarser level adds
    0.7 of its interpolated sum.  It stands for a trained network: the same work per
    application, and a multigrid-like Krylov convergence that needs no training here."""
    rng = np.random.default_rng(seed)
    ch = _channels(levels)
    first = np.linalg.qr(rng.standard_normal((ch[0], 1)))[0]
    down = [np.linalg.qr(rng.standard_normal((ch[l + 1], ch[l])))[0] for l in range(levels - 1)]

    def fill(role, l, ci, co):
        w = np.zeros((co, 9, ci))
        w[:, 4, :] = {"in": lambda: first, "out": lambda: first.T, "down": lambda: down[l],
                      "up": lambda: 0.7 * down[l].T}.get(role, lambda: np.eye(co))()
        return w

    return _theta(levels, fill)


def _network(h, w, batch, theta):
    n = _levels(h, w)
    net = learned.UNetPreconditioner(h, w, n, _channels(n), 1, 1, batch=batch)
    net.set_params(theta)
    return net


# ---- prepare and run ----------------------------------------------------------------------------

def prepare(case, seed):
    c = case
    dofs, settings, static = _inputs(c, seed)
    s = {"kind": c["kind"], "dofs": dofs, "settings": settings, "static": static}
    if c["kind"] == "newton":
        s["tol"] = 1e-11 if c["model"] == "cube" else 1e-10 if c["model"] == "panel" else 1e-12
        if c["precond"] == "learned":
            h, w = c["nx"] + 1, c["ny"] + 1
            s["net"] = _network(h, w, 1, _multilevel_weights(_levels(h, w), seed))
        s["prob"] = backend.get_problem(dofs, settings, static)
        return s
    if c["kind"] == "sensitivity":
        static.update({"linear tolerance": 1e-10})
        s["dofs"] = solver.solver(dofs, settings, static, newton_tol=1e-11)[0]
        return s
    prob = s["prob"] = backend.get_problem(dofs, settings, static)
    if c["kind"] == "assemble":
        if c["model"] == "vark":
            s["fields"] = [prob.to_device(settings[k]) for k in ("log coefficient", "source")]
            u = _waves(settings["node coordinates"], np.random.default_rng(seed + 1))
        else:
            u = _displacement(c, settings["node coordinates"], seed)
        s["u"] = prob.to_device(u.ravel())
        s["r"] = torch.empty_like(s["u"])
        s["vals"] = torch.empty(prob.nnz, dtype=torch.float64, device=prob.device)
        s["params"] = [prob.raw_params(i, settings) for i in range(len(prob.models))]
        return s
    s["vals"] = learned.tangent(prob)
    if c["kind"] == "pairs":
        gen = torch.Generator(device=prob.device).manual_seed(int(seed))
        s["rhs"] = torch.randn(prob.n_free, generator=gen, device=prob.device, dtype=torch.float64)
        return s
    free = torch.from_numpy(prob.free_dofs().astype(np.int64)).to(prob.device)
    h, w = c["nx"] + 1, c["ny"] + 1
    s["e"] = [torch.from_numpy(e).to(prob.device)[free] for e in _errors(c, seed)]
    s["res"] = [learned.spmv(prob, s["vals"], e) for e in s["e"]]
    s["net"] = _network(h, w, c["batch"], _starting_weights(_levels(h, w), seed))
    return s


def _errors(c, seed):
    """Solutions e of A e = r as training meets them: smooth, with a little of every wave length."""
    rng = np.random.default_rng(seed)
    x = _mesh(c["model"], c["nx"], c["ny"], c["nz"], c["skew"])[0]
    bubble = np.prod(np.sin(math.pi * x / x.max(axis=0)), axis=1)
    return [bubble * _waves(x, rng, 6, 30.0) + 1e-3 * rng.standard_normal(x.shape[0]) for _ in range(c["batch"])]


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    s = state
    if s["kind"] == "newton":
        if "net" in s:
            s["net"].attach(s["prob"])
        return {"dofs": solver.solver(s["dofs"], s["settings"], s["static"], newton_tol=s["tol"])[0]}
    if s["kind"] == "assemble":
        prob, stream = s["prob"], backend.current_stream()
        if "fields" in s:
            prob.bind_nodal_device(0, *s["fields"])
        else:
            for i, p in enumerate(s["params"]):
                prob.set_params(i, p)
        _native.call("apx_assemble_residual", prob.plan, _ptr(s["u"]), _ptr(s["r"]), stream)
        _native.call("apx_assemble_tangent", prob.plan, _ptr(s["u"]), _ptr(s["vals"]), _native.APX_FP64, stream)
        return {"residual": s["r"], "tangent": s["vals"]}
    if s["kind"] == "pairs":
        (r, e), = learned.solver_pairs(s["prob"], s["vals"], s["rhs"], checkpoints=(0,), tol=1e-12)
        return {"r": r, "e": e}
    if s["kind"] == "train":
        net, b = s["net"], len(s["e"])
        r_list, e_list = ((ctypes.c_void_p * b)(*[t.data_ptr() for t in ts]) for ts in (s["res"], s["e"]))
        loss = ctypes.c_double()
        _native.call("apx_unet_train_step", net.handle, s["prob"].plan, _ptr(s["vals"]), r_list, None, e_list, 2, 0.0,
                     ctypes.byref(loss), backend.current_stream())
        net.adam(5e-6)  # the rate that learned.fit ends with
        return {"loss": loss.value, "grads": net.get_grads()}
    g = implicit_diff.root_vjp(s["dofs"], s["settings"], s["static"], 2 * s["dofs"],
                               ["youngs modulus", "poisson ratio"])
    return {"dE": np.array([g["youngs modulus"]]), "dnu": np.array([g["poisson ratio"]])}


# ---- work ---------------------------------------------------------------------------------------

def work(case):
    """Bytes and flops that a pass cannot do without: its inputs and outputs once, and for the Krylov
    solves the matrix values and six vector passes per iteration (Jacobi-PCG needs about 2.6
    iterations per element along the longer side on these Poisson problems; the others as noted)."""
    c = case
    d = {"panel": 2, "q2": 2, "cube": 3}.get(c["model"], 1)
    nodes = (c["nx"] + 1) * (c["ny"] + 1) * (c["nz"] + 1) if c["model"] != "q2" else (2 * c["nx"] + 1) * (2 * c["ny"] + 1)
    elems = c["nx"] * c["ny"] * max(1, c["nz"])
    n = nodes * d
    row = {"cube": 81, "panel": 18, "q2": 32}.get(c["model"], 9)
    point = {"cube": 8 * 24 * 24 * 7, "panel": 4 * 64 * 7, "q2": 9 * 18 * 18 * 7}.get(c["model"], 4 * 16 * 3)
    once = n * 8 * 3 + nodes * len(str(d)) * 16
    assembly = elems * point
    if c["kind"] == "assemble":
        return {"bytes": once + n * row * 8, "flops": assembly}
    if c["kind"] == "train":
        p = sum(nodes / 4 ** l * ci * co * 18 for _, l, ci, co in _layers(_levels(c["nx"] + 1, c["ny"] + 1)))
        q = sum(nodes / 4 ** l * (ci + co) * 2 for _, l, ci, co in _layers(_levels(c["nx"] + 1, c["ny"] + 1)))
        return {"bytes": 3 * c["batch"] * q, "flops": 3 * c["batch"] * p}
    long = max(c["nx"], c["ny"], c["nz"])
    steps = {"panel": 5 * 60 * long, "q2": 80 * long, "cube": 3 * 5 * long}.get(c["model"], 2.6 * long)
    if c.get("precond") == "learned":
        steps = 4 * math.sqrt(long)
        layers = _layers(_levels(c["nx"] + 1, c["ny"] + 1))
        return {"bytes": once + steps * (n * (row + 6) * 8 + sum(nodes / 4 ** l * (ci + co) * 2 for _, l, ci, co in layers)),
                "flops": steps * sum(nodes / 4 ** l * ci * co * 18 for _, l, ci, co in layers)}
    values = 4 if c.get("precision") == "mixed" else 8
    return {"bytes": once + steps * n * (row * values + 6 * 8), "flops": assembly + steps * n * (row + 6) * 2}


# ---- results in 64 bits, by plain torch ---------------------------------------------------------

_DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
_GAUSS = {2: ((-1 / math.sqrt(3), 1 / math.sqrt(3)), (1.0, 1.0)),
          3: ((-math.sqrt(0.6), 0.0, math.sqrt(0.6)), (5 / 9, 8 / 9, 5 / 9))}


def _shape(model, xi):
    """Shape functions (NPE,) and reference gradients (NPE, dim) at the point xi."""
    x = torch.tensor(xi, dtype=torch.float64, requires_grad=True)
    quad = lambda t: (0.5 * t * (t - 1), 1 - t * t, 0.5 * t * (t + 1))  # noqa: E731
    if model == "q2":
        a, b = quad(x[0]), quad(x[1])
        N = torch.stack([a[i] * b[j] for i, j in zip((0, 2, 2, 0, 1, 2, 1, 0, 1), (0, 0, 2, 2, 0, 1, 2, 1, 1))])
    elif len(xi) == 3:
        N = torch.stack([(1 + i * x[0]) * (1 + j * x[1]) * (1 + k * x[2]) / 8 for k in (-1, 1)
                         for i, j in ((-1, -1), (1, -1), (1, 1), (-1, 1))])
    else:
        N = torch.stack([(1 + i * x[0]) * (1 + j * x[1]) / 4 for i, j in ((-1, -1), (1, -1), (1, 1), (-1, 1))])
    dN = torch.stack([torch.autograd.grad(n, x, retain_graph=True)[0] for n in N])
    return N.detach().to(_DEVICE), dN.to(_DEVICE)


def _inverse(F):
    """Determinant and inverse of (..., 2, 2) or (..., 3, 3)."""
    if F.shape[-1] == 2:
        adj = torch.stack([torch.stack([F[..., 1, 1], -F[..., 0, 1]], -1), torch.stack([-F[..., 1, 0], F[..., 0, 0]], -1)], -2)
        det = F[..., 0, 0] * F[..., 1, 1] - F[..., 0, 1] * F[..., 1, 0]
    else:
        a, b, c = F[..., 0, :], F[..., 1, :], F[..., 2, :]
        adj = torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)], -1)
        det = (a * adj[..., :, 0]).sum(-1)
    return det, adj / det[..., None, None]


class _NoValue(Exception):
    """The plain solve did not converge: no value to compare with."""


def _times(A, x):
    V, C = A
    return (V * x[C]).sum(0)


class _Exact:
    """Residual, reduced tangent and solves of a case in FP64 on the GPU."""

    def __init__(self, c, settings):
        self.c, self.s = c, settings
        coords, sets, mask, _ = _mesh(c["model"], c["nx"], c["ny"], c["nz"], c["skew"])
        self.x = torch.from_numpy(coords).to(_DEVICE)
        self.conn = torch.from_numpy(sets[0]).to(_DEVICE)
        self.d = 1 if mask.ndim == 1 else mask.shape[1]
        self.mask = torch.from_numpy(mask.ravel().copy()).to(_DEVICE)
        self.n = self.mask.numel()
        self.free = torch.nonzero(~self.mask).ravel()
        self.dof = (self.conn[:, :, None] * self.d + torch.arange(self.d, device=_DEVICE)).flatten(1)
        t, w = _GAUSS[3 if c["model"] == "q2" else 2]
        dim = coords.shape[1]
        grid = [[]]
        for _ in range(dim):
            grid = [p + [i] for p in grid for i in range(len(t))]
        self.points = [(*_shape(c["model"], [t[i] for i in p]), math.prod(w[i] for i in p)) for p in grid]
        self.load = self._load(sets)
        if c["model"] in ("panel", "cube"):
            self.lam, self.mu = settings["lam"], settings["mu"]
        elif c["model"] == "q2":
            E, nu = settings["youngs modulus"], settings["poisson ratio"]
            self.lam, self.mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
        elif c["model"] == "vark":
            self.g, self.f = (torch.from_numpy(settings[k]).to(_DEVICE) for k in ("log coefficient", "source"))

    def _load(self, sets):
        out = torch.zeros(self.n, dtype=torch.float64, device=_DEVICE)
        if len(sets) == 1:
            return out
        lines, x = torch.from_numpy(sets[1]).to(_DEVICE), self.x
        t = self.s["load multiplier"] * (1.0 / 16.0 if self.c["model"] == "panel" else 1.0)
        length = (x[lines[:, 1]] - x[lines[:, 0]]).norm(dim=1)
        for k, part in enumerate((0.5, 0.5) if lines.shape[1] == 2 else (1 / 6, 1 / 6, 2 / 3)):
            out.index_add_(0, lines[:, k] * 2 + 1, -t * part * length)
        return out

    def elements(self, u, at, tangent):
        """Element residuals and matrices of the elements `at`."""
        c, d, conn = self.c, self.d, self.conn[at]
        xe, ue = self.x[conn], u.view(-1, d)[conn]
        r = K = 0.0
        for N, dN, w in self.points:  # sums of products: batches of tiny matrix products are slow
            det, inv = _inverse((xe[:, :, :, None] * dN[:, None, :]).sum(1))
            G = (dN[:, :, None] * inv[:, None]).sum(2)
            w = w * det
            GG = (G[:, :, None] * G[:, None]).sum(3)
            if d == 1:
                k, grad = 1.0, (ue * G).sum(1)
                if c["model"] == "vark":
                    k, b = torch.exp(self.g[conn] @ N)[:, None], self.f[conn] @ N
                else:
                    amp, freq, cx, cy = SOURCE
                    q = (N[:, None] * xe).sum(1)
                    y = q - torch.tensor([cx, cy], dtype=torch.float64, device=_DEVICE)
                    b = amp * (torch.sin(freq * (q * q).sum(1)) - torch.cos(freq * (y * y).sum(1)))
                r = r + w[:, None] * (k * (G * grad[:, None]).sum(2) - b[:, None] * N)
                if tangent:
                    K = K + (w[:, None] * k)[:, :, None] * GG
                continue
            eye = torch.eye(d, dtype=torch.float64, device=_DEVICE)
            F = (ue[:, :, :, None] * G[:, :, None]).sum(1) + eye
            J, Fi = _inverse(F)
            H = (Fi[:, None] * G[:, :, :, None]).sum(2)
            c1 = self.mu - 0.5 * self.lam * (J * J - 1)
            FG = (F[:, None] * G[:, :, None]).sum(3)
            r = r + (w[:, None, None] * (self.mu * FG - c1[:, None, None] * H)).flatten(1)
            if tangent:  # (element, a, i, b, k)
                wide = lambda t: t[:, None, None, None, None]  # noqa: E731
                k = self.mu * GG[:, :, None, :, None] * eye[:, None, :]
                k = k + wide(c1) * H[:, :, None, None, :] * H.transpose(1, 2)[:, None, :, :, None]
                k = k + wide(self.lam * J * J) * H[:, :, :, None, None] * H[:, None, None]
                K = K + (wide(w) * k).flatten(3).flatten(1, 2)
        return r, K

    def assemble(self, u, tangent=True):
        r = self.load.clone()
        if tangent and not hasattr(self, "slot"):
            place = torch.full((self.n,), -1, dtype=torch.int64, device=_DEVICE)
            place[self.free] = torch.arange(self.free.numel(), device=_DEVICE)
            rd = place[self.dof]
            key = rd[:, :, None] * self.free.numel() + rd[:, None, :]
            key[(rd < 0)[:, :, None] | (rd < 0)[:, None, :]] = -1
            uniq, slot = torch.unique(key.ravel(), return_inverse=True)
            skip = int(uniq[0] < 0)
            self.key, self.slot = uniq[skip:], slot.view(key.shape) - skip
        vals = torch.zeros(self.key.numel(), dtype=torch.float64, device=_DEVICE) if tangent else None
        for lo in range(0, self.conn.shape[0], 1 << 16):
            at = slice(lo, lo + (1 << 16))
            re, Ke = self.elements(u, at, tangent)
            r.index_add_(0, self.dof[at].ravel(), re.ravel())
            if tangent:
                slot = self.slot[at].ravel()
                kept = slot >= 0  # (thousands of atomic additions to one spare slot would take minutes)
                vals.index_add_(0, slot[kept], Ke.ravel()[kept])
        return r, vals

    def matrix(self, vals):
        """The reduced matrix as (values, columns), each (longest row, rows), and its diagonal."""
        m = self.free.numel()
        rows = torch.div(self.key, m, rounding_mode="floor")
        count = torch.bincount(rows, minlength=m)
        k = torch.arange(self.key.numel(), device=_DEVICE) - (torch.cumsum(count, 0) - count)[rows]
        V = torch.zeros(int(count.max()), m, dtype=torch.float64, device=_DEVICE)
        C = torch.zeros(V.shape, dtype=torch.int64, device=_DEVICE)
        V[k, rows], C[k, rows] = vals, self.key % m
        diag = torch.zeros(m, dtype=torch.float64, device=_DEVICE)
        on = self.key % m == rows
        diag[rows[on]] = vals[on]
        return (V, C), diag

    def solve(self, A, diag, b, tol=1e-10):
        """Jacobi-PCG, the residual refreshed once so that the error ends at the rounding of A x."""
        x = torch.zeros_like(b)
        for _ in range(2):
            r = b - _times(A, x)
            target = tol * float(r.norm())
            z = r / diag
            p, rz, dx = z.clone(), r @ z, torch.zeros_like(b)
            for k in range(20000):
                q = _times(A, p)
                a = rz / (p @ q)
                dx += a * p
                r -= a * q
                if k % 50 == 49:
                    size = float(r.norm())
                    if size <= target:
                        break
                    if not math.isfinite(size) or k == 19999:
                        raise _NoValue
                z = r / diag
                new = r @ z
                p = z + (new / rz) * p
                rz = new
            x += dx
        return x

    def newton(self, u):
        u = u.clone()
        v = self.s["dirichlet conditions"]
        u[self.mask] = torch.from_numpy((v["u"] if isinstance(v, dict) else v).ravel()).to(_DEVICE)[self.mask]
        for _ in range(1 if self.d == 1 else 8):
            r, vals = self.assemble(u)
            A, diag = self.matrix(vals)
            dx = self.solve(A, diag, -r[self.free])
            u[self.free] += dx
            if float(dx.norm()) < 1e-13 * float(u.norm()):
                break
        return u


def _transfer(m):
    """Bilinear interpolation from ceil(m / 2) to m nodes."""
    P = torch.zeros(m, (m + 1) // 2, dtype=torch.float64, device=_DEVICE)
    i = torch.arange(m, device=_DEVICE)
    P[i[::2], i[::2] // 2] = 1.0
    P[i[1::2], i[1::2] // 2] = 0.5
    right = i[1::2][i[1::2] // 2 + 1 < P.shape[1]]
    P[right, right // 2 + 1] = 0.5
    return P


def _network64(theta, x, levels):
    """The network's output for images x (batch, 1, h, w), in FP64."""
    W = {}
    for role, l, ci, co, cop, wk, off in list(_layout(levels))[:-1]:
        w = theta[off:off + cop * wk].view(cop, wk)[:co, :9 * ci].reshape(co, 3, 3, ci)
        W[role, l] = w.permute(0, 3, 1, 2)
    conv = lambda k, t: torch.nn.functional.conv2d(t, W[k], padding=1)  # noqa: E731
    a, skips, ps = conv(("in", 0), x), [], []
    for l in range(levels - 1):
        skips.append(conv(("e", l), a))
        ps.append((_transfer(a.shape[2]), _transfer(a.shape[3])))
        a = conv(("down", l), ps[l][0].T @ skips[l] @ ps[l][1])
    u = conv(("b", levels - 1), a)
    for l in range(levels - 2, -1, -1):
        u = conv(("d", l), skips[l] + ps[l][0] @ conv(("up", l), u) @ ps[l][1].T)
    return conv(("out", 0), u)


def _train64(c, seed, ex):
    """Loss and gradients of a training step (relative A-norm error, Jacobi scaling)."""
    _, vals = ex.assemble(torch.zeros(ex.n, dtype=torch.float64, device=_DEVICE))
    A, diag = ex.matrix(vals)
    h, w, scale = c["nx"] + 1, c["ny"] + 1, diag.abs().rsqrt()
    levels = _levels(h, w)
    theta = torch.from_numpy(_starting_weights(levels, seed)).to(_DEVICE).double().requires_grad_()
    loss, sign = 0.0, math.copysign(1.0, float(diag[0]))
    grad = torch.zeros_like(theta)
    for e in _errors(c, seed):
        e = torch.from_numpy(e).to(_DEVICE)[ex.free]
        r = _times(A, e)
        s = (scale * r).square().mean().sqrt()
        x = torch.zeros(ex.n, dtype=torch.float64, device=_DEVICE)
        x[ex.free] = scale * r / s
        with torch.backends.cudnn.flags(enabled=False):
            z = scale * s * _network64(theta, x.view(1, 1, h, w), levels).ravel()[ex.free]
            zd = z.detach()
            res, energy = r - _times(A, zd), sign * (e @ r)
            loss += float(-sign * ((zd - e) @ res) / energy) / c["batch"]
            grad += torch.autograd.grad(z, theta, -2.0 * sign * res / energy / c["batch"])[0]
    return {"loss": loss, "grads": grad.float().cpu().numpy()}


def exact(case, seed):
    try:
        return _exact(case, seed)
    except _NoValue:
        return None


def _exact(c, seed):
    dofs, settings, _ = _inputs(c, seed)
    ex = _Exact(c, settings)
    if c["kind"] == "newton":
        if c["model"] == "panel" and c["nx"] * c["ny"] > 6000:
            return None
        start = dofs["u"] if isinstance(dofs, dict) else dofs
        u = ex.newton(torch.from_numpy(start.ravel()).to(_DEVICE)).cpu().numpy()
        return {"dofs": {"u": u} if isinstance(dofs, dict) else u}
    if c["kind"] == "assemble":
        if c["model"] == "vark":
            u = _waves(settings["node coordinates"], np.random.default_rng(seed + 1))
        else:
            u = _displacement(c, settings["node coordinates"], seed)
        r, vals = ex.assemble(torch.from_numpy(u.ravel()).to(_DEVICE))
        return {"residual": r, "tangent": vals}
    if c["kind"] == "pairs":
        _, vals = ex.assemble(torch.zeros(ex.n, dtype=torch.float64, device=_DEVICE))
        gen = torch.Generator(device=_DEVICE).manual_seed(int(seed))
        b = torch.randn(ex.free.numel(), generator=gen, device=_DEVICE, dtype=torch.float64)
        return {"r": b, "e": ex.solve(*ex.matrix(vals), b)}
    if c["kind"] == "train":
        return _train64(c, seed, ex)
    u = ex.newton(torch.zeros(ex.n, dtype=torch.float64, device=_DEVICE))
    _, vals = ex.assemble(u)
    lam, mu, load = ex.lam, ex.mu, ex.load
    w = torch.zeros_like(u)
    w[ex.free] = ex.solve(*ex.matrix(vals), -2 * u[ex.free])
    ex.load = torch.zeros_like(load)
    parts = []
    for ex.lam, ex.mu in ((1.0, 0.0), (0.0, 1.0)):  # the residual is linear in (lam, mu)
        parts.append(float(w @ ex.assemble(u, tangent=False)[0]))
    E, nu = settings["youngs modulus"], settings["poisson ratio"]
    a, b = (1 + nu) * (1 - 2 * nu), 1 + nu
    dlam, dmu = E / a + E * nu * (1 + 4 * nu) / a ** 2, -E / (2 * b * b)
    return {"dE": np.array([parts[0] * lam / E + parts[1] * mu / E]), "dnu": np.array([parts[0] * dlam + parts[1] * dmu])}
