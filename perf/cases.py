"""The work that programs on this framework have it do, for timing and for comparing results.

The listed cases are the five benchmark configurations of ``phasefield_amd.prm`` (Allen-Cahn
2D, Cahn-Hilliard 3D, Poisson 3D, the Allen-Cahn adjoint, the coupled precipitate model), the
two reference applications that ``bench.py`` measures beside them (linear elasticity, implicit
Allen-Cahn), and small or ragged meshes of the same models.  `draw` gives more of each kind:
meshes from a few thousand nodes to the largest listed one, cell counts that no tile divides,
unequal extents, both arithmetic precisions and the preconditioners the models are run with.

A state is a context with its fields in place; `run` starts from those fields every time, so
it can be repeated.  `exact` restates each model in plain torch and FP64: on these uniform
meshes with collocated quadrature the assembled operators are M (r(u) + beta L u), with M the
lumped mass and L the line stencils of `_Axis`; elasticity is assembled cell by cell.
"""

from __future__ import annotations

import math

import torch

from phasefield_amd import Context, prm
from phasefield_amd.capi import (AGE_LATEST, FP32, FP64, OP_LHS, OP_RHS, SCALE_NONE)

DT_AC2D, DT_CH, DT_PRECIPITATE, DT_ADJOINT, DT_IMPLICIT = 0.005, 1e-4, 5e-3, 0.01, 0.01
SPACING = 100.0 / 64.0  # cell edge of the elasticity application's mesh
APPLICATIONS = 4        # operator applications in a pass of the apply kinds


# ------------------------------------------------------------------------------- the cases
def listed():
    return [
        # Allen-Cahn 2D at the benchmark size: 66k nodes, a launch per increment, so latency
        # and launch count are what a user of small 2D problems waits for.
        {"name": "ac2d_256", "kind": "ac2d", "nx": 256, "ny": 256, "steps": 100},
        # Cahn-Hilliard 3D Q2 at the benchmark size, the flagship increment loop.
        {"name": "ch3d_64", "kind": "ch3d", "nx": 64, "ny": 64, "nz": 64, "steps": 20},
        # The coupled precipitate model at the benchmark size: three fields, memory bound.
        {"name": "precipitate_192", "kind": "precipitate", "nx": 192, "ny": 192, "nz": 192,
         "steps": 10, "single": False},
        # The same model on an uneven box with FP32 arithmetic on the FP64 state.
        {"name": "precipitate_single_ragged", "kind": "precipitate", "nx": 150, "ny": 77,
         "nz": 51, "steps": 20, "single": True},
        # The Poisson operator at the benchmark size, as a user's own Krylov loop applies it.
        {"name": "poisson_apply_128", "kind": "poisson_apply", "nx": 128, "ny": 128, "nz": 128,
         "single": False},
        # ... on an uneven box in FP32 (a preconditioner's precision).
        {"name": "poisson_apply_single_ragged", "kind": "poisson_apply", "nx": 90, "ny": 54,
         "nz": 70, "single": True},
        # Time to solution of the Poisson configuration: CG with a geometric-multigrid V-cycle,
        # FP32 levels under the FP64 outer iteration.
        {"name": "poisson_gmg_128", "kind": "poisson_gmg", "nx": 1, "ny": 1, "nz": 1,
         "refinement": 7, "single": True},
        # A small 2D solve: every kernel is far below the chip's size, launches count.
        {"name": "poisson_gmg_2d_64", "kind": "poisson_gmg", "nx": 1, "ny": 1, "nz": 0,
         "refinement": 6, "single": False},
        # Linear elasticity at the reference application's mesh: the operator alone (three
        # coupled fields, the generic cell path) ...
        {"name": "elasticity_apply_64", "kind": "elasticity_apply", "nx": 64, "ny": 64,
         "nz": 64},
        # ... and the reference application's solve (CG without a preconditioner) on a smaller,
        # uneven bar.
        {"name": "elasticity_cg_bar", "kind": "elasticity_cg", "nx": 40, "ny": 24, "nz": 17,
         "chebyshev": False},
        # Gradients of an Allen-Cahn run: backward sweep with checkpoints.
        {"name": "adjoint_128", "kind": "adjoint", "nx": 128, "ny": 128, "nz": 128, "steps": 20,
         "every": 10, "single": False},
        # Implicit Allen-Cahn 2D at the reference application's mesh: Newton with CG.
        {"name": "ac2d_implicit_256", "kind": "ac2d_implicit", "nx": 256, "ny": 256, "steps": 5,
         "gmg": False},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _box(rng, low, high, most):
    """Cell counts in [low, high] per axis, at most `most` cells in all."""
    while True:
        n = [_log_int(rng, low, high) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most:
            return {"nx": n[0], "ny": n[1], "nz": n[2]}


def draw(rng):
    kind = rng.choice(["ac2d", "ch3d", "precipitate", "poisson_apply", "poisson_gmg",
                       "elasticity_apply", "elasticity_cg", "adjoint", "ac2d_implicit"])
    if kind == "ac2d":
        return {"kind": kind, "nx": _log_int(rng, 24, 900), "ny": _log_int(rng, 24, 900),
                "steps": rng.randint(20, 100)}
    if kind == "ch3d":
        return {"kind": kind, **_box(rng, 8, 96, 64 ** 3), "steps": rng.randint(6, 20)}
    if kind == "precipitate":
        return {"kind": kind, **_box(rng, 16, 256, 192 ** 3), "steps": rng.randint(4, 20),
                "single": rng.random() < 0.5}
    if kind == "poisson_apply":
        return {"kind": kind, **_box(rng, 8, 200, 128 ** 3), "single": rng.random() < 0.5}
    if kind == "poisson_gmg":
        refinement = rng.randint(3, 5)
        most = {3: 12, 4: 6, 5: 3}[refinement]
        flat = rng.random() < 0.4
        return {"kind": kind, "nx": rng.randint(1, most), "ny": rng.randint(1, most),
                "nz": 0 if flat else rng.randint(1, most), "refinement": refinement,
                "single": rng.random() < 0.5}
    if kind == "elasticity_apply":
        return {"kind": kind, **_box(rng, 4, 96, 64 ** 3)}
    if kind == "elasticity_cg":
        return {"kind": kind, **_box(rng, 4, 40, 40 * 24 * 17), "chebyshev": rng.random() < 0.4}
    if kind == "adjoint":
        steps = rng.randint(8, 20)
        return {"kind": kind, **_box(rng, 12, 160, 128 ** 3), "steps": steps,
                "every": rng.randint(3, steps), "single": rng.random() < 0.4}
    if rng.random() < 0.3:
        return {"kind": kind, "nx": rng.randint(2, 12), "ny": rng.randint(2, 12),
                "refinement": 4, "steps": rng.randint(1, 3), "gmg": True}
    return {"kind": kind, "nx": _log_int(rng, 24, 400), "ny": _log_int(rng, 24, 400),
            "steps": rng.randint(1, 5), "gmg": False}


# ------------------------------------------------------------------- lattices and operators
_MODELS = {  # kind -> (degree, periodic)
    "ac2d": (1, True), "ch3d": (2, True), "precipitate": (1, True), "poisson_apply": (2, False),
    "poisson_gmg": (2, False), "elasticity_apply": (2, False), "elasticity_cg": (2, False),
    "adjoint": (1, True), "ac2d_implicit": (1, False),
}


def _cells(case):
    """Cells per axis, x first."""
    n = [case["nx"], case["ny"]] + ([case["nz"]] if case.get("nz") else [])
    return [k << case.get("refinement", 0) for k in n]


def _size(case):
    """Edge lengths of the domain: the benchmark spacing of each model."""
    cells = _cells(case)
    h = {"ac2d": 100.0 / 256.0, "ch3d": 1.0, "precipitate": 1.0, "adjoint": 1.0,
         "elasticity_apply": SPACING, "elasticity_cg": SPACING,
         "ac2d_implicit": 100.0 / 256.0}.get(case["kind"], 1.0 / max(cells))
    return [h * n for n in cells]


def _nodes(case):
    """Stored nodes per axis, x first."""
    degree, periodic = _MODELS[case["kind"]]
    return [degree * n + (0 if periodic else 1) for n in _cells(case)]


def _shape(case):
    return tuple(reversed(_nodes(case)))


class _Axis:
    """One axis of the lattice: neighbour indices (wrapped, or mirrored at the ends), taps by
    node and lumped masses."""

    def __init__(self, n, h, degree, periodic, device):
        i = torch.arange(n, device=device)
        self.n, self.degree = n, degree
        self.near = {}
        for o in range(1, degree + 1):
            pair = []
            for j in (i - o, i + o):
                if periodic:
                    j = j % n
                else:
                    j = j.abs()
                    j = torch.where(j > n - 1, 2 * (n - 1) - j, j)
                pair.append(j)
            self.near[o] = pair
        if degree == 2:
            odd = (i % 2 == 1).double()
            even = 1.0 - odd
            self.taps = [(14.0 * even + 8.0 * odd) / h ** 2, (-8.0 * even - 4.0 * odd) / h ** 2,
                         even / h ** 2]
            self.mass = (even / 3.0 + odd * 2.0 / 3.0) * h
        else:
            one = torch.ones(n, dtype=torch.float64, device=device)
            self.taps = [2.0 * one / h ** 2, -one / h ** 2]
            self.mass = one * h
        if not periodic:
            self.mass[0] *= 0.5
            self.mass[-1] *= 0.5

    def dense(self):
        """The axis' L as a matrix."""
        m = torch.diag(self.taps[0])
        rows = torch.arange(self.n, device=m.device)
        for o in range(1, self.degree + 1):
            for j in self.near[o]:
                m.index_put_((rows, j), self.taps[o], accumulate=True)
        return m


class _Lattice:
    def __init__(self, case, device):
        degree, periodic = _MODELS[case["kind"]]
        cells, size = _cells(case), _size(case)
        self.dim = len(cells)
        self.axes = [_Axis(degree * n + (0 if periodic else 1), s / n, degree, periodic, device)
                     for n, s in zip(cells, size)]

    def _along(self, v, d):
        return v.reshape([-1 if k == self.dim - 1 - d else 1 for k in range(self.dim)])

    def lap(self, u):
        """L u = M^{-1} K u (positive: minus the Laplacian)."""
        out = None
        for d, ax in enumerate(self.axes):
            t = self.dim - 1 - d
            term = self._along(ax.taps[0], d) * u
            for o, (lo, hi) in ax.near.items():
                term += self._along(ax.taps[o], d) * (u.index_select(t, lo) + u.index_select(t, hi))
            out = term if out is None else out + term
        return out

    def mass(self):
        m = self._along(self.axes[0].mass, 0)
        for d in range(1, self.dim):
            m = m * self._along(self.axes[d].mass, d)
        return m


# ------------------------------------------------------------------------ inputs and states
class _Device:
    """A field of a context, described so that torch can take it as a tensor.  The tensor keeps
    this object, and this object the context that owns the memory."""

    def __init__(self, ctx, ptr, shape):
        self.owner = ctx
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape),
                                         "typestr": "<f8", "version": 3, "strides": None}


def _field(state, field, age):
    """The context's own buffer of a field state.  A context has a few buffers per field and
    swaps them as it steps; each is wrapped once."""
    ptr = state["ctx"].field_device_ptr(field, age)
    if ptr not in state["views"]:
        state["views"][ptr] = torch.as_tensor(_Device(state["ctx"], ptr, state["shape"]), device="cuda")
    return state["views"][ptr]


def _generator(seed, device):
    return torch.Generator(device=device).manual_seed(1000003 * (int(seed) + 1))


def _coordinates(case, device):
    degree, _ = _MODELS[case["kind"]]
    xs = []
    nodes, cells, size = _nodes(case), _cells(case), _size(case)
    for d in range(len(nodes)):
        x = torch.arange(nodes[d], dtype=torch.float64, device=device) * size[d] / (degree * cells[d])
        xs.append(x.reshape([-1 if k == len(nodes) - 1 - d else 1 for k in range(len(nodes))]))
    return xs


def _blobs(case, gen, device, count, radii, width):
    """Smooth spheres in the box, as the models' initial conditions nucleate them (smaller
    ones in a small box)."""
    xs, size = _coordinates(case, device), _size(case)
    scale = min(1.0, 0.25 * min(size) / radii[1])
    out = torch.zeros(_shape(case), dtype=torch.float64, device=device)
    draws = torch.rand((count, 4), dtype=torch.float64, device=device, generator=gen).cpu().tolist()
    for row in draws:
        r2 = 0.0
        for d, x in enumerate(xs):
            dx = x - row[d] * size[d]
            dx = dx - size[d] * torch.round(dx / size[d])
            r2 = r2 + dx * dx
        radius = scale * (radii[0] + (radii[1] - radii[0]) * row[3])
        out += 0.5 * (1.0 - torch.tanh((torch.sqrt(r2) - radius) / width))
    return out


def _uniform(case, gen, device, low, high, fields=1, dtype=torch.float64):
    shape = _shape(case) if fields == 1 else (fields,) + _shape(case)
    return torch.rand(shape, dtype=torch.float64, device=device, generator=gen).mul_(high - low).add_(low).to(dtype)


def _inputs(case, seed, device):
    """The arrays (and material constants) of a case, from the seed alone."""
    gen, kind = _generator(seed, device), case["kind"]
    if kind in ("ac2d", "adjoint"):
        phi = _blobs(case, gen, device, 8, (5.0, 15.0), 1.0)
        phi = phi + _uniform(case, gen, device, -0.05, 0.05)
        if kind == "ac2d":
            return {"phi": phi}
        # the gradient of a misfit to another state
        target = _blobs(case, gen, device, 8, (5.0, 15.0), 1.0)
        target = target + _uniform(case, gen, device, -0.05, 0.05)
        return {"phi": phi.contiguous(), "lam": (phi - target).contiguous()}
    if kind == "ch3d":
        c = _uniform(case, gen, device, 0.49, 0.51)
        mu = 2.0 * c * (1.0 - c) * (1.0 - 2.0 * c) + _Lattice(case, device).lap(c)
        return {"c": c, "mu": mu}
    if kind == "precipitate":
        c = _uniform(case, gen, device, 0.29, 0.31)
        eta = _blobs(case, gen, device, 20, (4.0, 4.0), 1.0).clamp_(max=1.0)
        return {"c": c, "eta": eta, "mu": _precipitate_mu(c, eta, _Lattice(case, device))}
    if kind == "poisson_gmg":
        return {"f": torch.randn(_shape(case), dtype=torch.float64, device=device, generator=gen)}
    if kind == "poisson_apply":
        return {"u": _uniform(case, gen, device, -1.0, 1.0,
                              dtype=torch.float32 if case["single"] else torch.float64)}
    if kind == "elasticity_apply":
        return {"u": _uniform(case, gen, device, -1.0, 1.0, fields=3), "E": 2.0, "nu": 0.3}
    if kind == "elasticity_cg":
        e, nu = torch.rand(2, dtype=torch.float64, device=device, generator=gen).cpu().tolist()
        return {"E": 1.0 + 2.0 * e, "nu": 0.28 + 0.04 * nu}
    return {"n": _blobs(case, gen, device, 12, (10.0, 20.0), 1.5).clamp_(max=1.0)}


def _mesh_text(text, case):
    """`text` on the case's mesh: its extents, subdivisions and refinement in place of the
    cube the parameter helpers write."""
    n = [case["nx"], case["ny"]] + ([case["nz"]] if case.get("nz") else [])
    size, out = _size(case), []
    for line in text.splitlines():
        words = line.split()
        axis = len(words) > 3 and words[0] == "set" and words[1] in ("x", "y", "z")
        if axis and words[2] == "size":
            line = "  set %s size = %r" % (words[1], size["xyz".index(words[1])])
        elif axis and words[2] == "subdivisions":
            line = "  set %s subdivisions = %d" % (words[1], n["xyz".index(words[1])])
        elif line.startswith("set global refinement"):
            line = "set global refinement = %d" % case.get("refinement", 0)
        out.append(line)
    return "\n".join(out) + "\n"


def _context(case, given):
    kind, many = case["kind"], 10 ** 6  # many: no output increment falls into a pass
    if kind == "ac2d":
        app, text = "allen_cahn_2d_q1", prm.allen_cahn(dim=2, steps=many, dt=DT_AC2D)
    elif kind == "ch3d":
        app, text = "cahn_hilliard_3d_q2", prm.cahn_hilliard(steps=many, dt=DT_CH)
    elif kind == "precipitate":
        app, text = "precipitate_3d_q1", prm.precipitate(steps=many, dt=DT_PRECIPITATE)
    elif kind == "adjoint":
        app = "allen_cahn_3d_q1"
        text = prm.allen_cahn(dim=3, steps=many, dt=DT_ADJOINT)
    elif kind in ("poisson_apply", "poisson_gmg"):
        dim = len(_cells(case))
        app = "poisson_%dd_q2" % dim
        text = prm.poisson(dim=dim, mg_depth=max(1, case.get("refinement", 0)),
                           preconditioner="GMG" if kind == "poisson_gmg" else "None",
                           level_precision="single" if case["single"] else "double")
    elif kind in ("elasticity_apply", "elasticity_cg"):
        app = "mechanics_3d_q2"
        text = prm.mechanics(E=given["E"], nu=given["nu"],
                             preconditioner="Chebyshev" if case.get("chebyshev") else None)
    else:
        # solver tolerances below the reference application's, so that the new state is a
        # result of the inputs and not of where an iteration happened to stop
        app = "allen_cahn_implicit_2d_q1"
        text = prm.allen_cahn_implicit(steps=many, outputs=1, dt=DT_IMPLICIT,
                                       linear_tolerance=1e-9, newton_tolerance=1e-8,
                                       preconditioner="GMG" if case["gmg"] else None,
                                       mg_depth=case["refinement"] if case["gmg"] else None)
    return Context(app, _mesh_text(text, case))


def prepare(case, seed):
    given = _inputs(case, seed, "cuda")
    ctx = _context(case, given)
    state = {"case": case, "ctx": ctx, "given": given, "views": {}, "shape": _shape(case)}
    kind = case["kind"]
    if kind == "precipitate" and case["single"]:
        ctx.set_option("explicit_precision", "single")
    elif kind in ("poisson_apply", "elasticity_apply"):
        ctx.set_option("synchronize", "0")
        state["work"] = [torch.empty_like(given["u"]) for _ in range(2)]
    elif kind == "poisson_gmg":
        _field(state, 1, 0).copy_(given["f"])
        ctx.set_time(1, 0.0)
        b = torch.empty_like(given["f"])
        ctx.apply_operator(1, OP_RHS, SCALE_NONE, FP64, 0, b.data_ptr())
        ctx.set_option("linear_tolerance", 1e-8 * float(torch.linalg.vector_norm(b)))
        ctx.set_option("linear_initial_guess", "zero")
    elif kind in ("elasticity_cg", "ac2d_implicit"):
        ctx.set_time(1, 0.0)
        ctx.set_option("linear_initial_guess", "zero")
    elif kind == "adjoint":
        state["grad"] = torch.empty_like(given["phi"])
    torch.cuda.synchronize()
    return state


def _steps(state, fields, dt):
    """The fields' states (field, name, age) put in place, then the case's increments."""
    ctx = state["ctx"]
    for field, name, age in fields:
        _field(state, field, age).copy_(state["given"][name])
    ctx.set_time(1, dt)
    if ctx.run(state["case"]["steps"]) != 0:
        raise RuntimeError("the run stopped")
    return {name: _field(state, field, AGE_LATEST) for field, name, _ in fields}


def run(state):
    case, ctx, given = state["case"], state["ctx"], state["given"]
    kind = case["kind"]
    if kind == "ac2d":
        return _steps(state, [(0, "phi", 1)], DT_AC2D)
    if kind == "ch3d":
        return _steps(state, [(0, "c", 1), (1, "mu", 1)], DT_CH)
    if kind == "precipitate":
        return _steps(state, [(0, "c", 1), (1, "mu", 1), (2, "eta", 1)], DT_PRECIPITATE)
    if kind == "ac2d_implicit":
        return _steps(state, [(0, "n", 1)], DT_IMPLICIT)
    if kind in ("poisson_apply", "elasticity_apply"):
        src = given["u"]
        precision = FP32 if case.get("single") else FP64
        for k in range(APPLICATIONS):
            dst = state["work"][k % 2]
            ctx.apply_operator(1, OP_LHS, SCALE_NONE, precision, src.data_ptr(), dst.data_ptr())
            src = dst
        ctx.synchronize()
        return src
    if kind == "poisson_gmg":
        if not ctx.linear_solve(1).converged:
            raise RuntimeError("the solve did not converge")
        return _field(state, 0, 0)
    if kind == "elasticity_cg":
        if not ctx.linear_solve(1).converged:
            raise RuntimeError("the solve did not converge")
        return [_field(state, f, 0) for f in range(3)]
    dL, dkappa = ctx.adjoint_vjp(given["phi"].data_ptr(), given["lam"].data_ptr(), 1.0, 1.5,
                                 case["steps"], case["every"], FP32 if case["single"] else FP64,
                                 state["grad"].data_ptr())
    return {"dL": dL, "dkappa": dkappa, "dphi0": state["grad"]}


# ---------------------------------------------------------------------------- what it costs
def work(case):
    """Bytes and operations of a pass, each array of each step or application once.  Solves
    are counted with the iterations they take (about 5 V-cycles, 14 CG steps per cell of the
    longest edge, 3 Newton updates of 10 CG steps), a step with what its operator and vectors need."""
    n, kind = 1.0, case["kind"]
    for k in _nodes(case):
        n *= k
    if kind == "ac2d":
        return {"bytes": 16 * n * case["steps"], "flops": 20 * n * case["steps"]}
    if kind == "ch3d":
        return {"bytes": 40 * n * case["steps"], "flops": 60 * n * case["steps"]}
    if kind == "precipitate":
        return {"bytes": 72 * n * case["steps"], "flops": 100 * n * case["steps"]}
    if kind == "poisson_apply":
        size = 4 if case["single"] else 8
        return {"bytes": 2 * size * n * APPLICATIONS, "flops": 25 * n * APPLICATIONS}
    if kind == "elasticity_apply":
        # the assembled operator's 3 x 3 coupled rows, by sum factorization
        return {"bytes": 48 * n * APPLICATIONS, "flops": 330 * n * APPLICATIONS}
    if kind == "poisson_gmg":
        # a V-cycle: 4 + 4 smoothing steps of 4 arrays on levels that add up to 8/7 (4/3) n,
        # a residual and the transfers; an outer step: 8 FP64 arrays
        levels = 8.0 / 7.0 if len(_cells(case)) == 3 else 4.0 / 3.0
        size = 4 if case["single"] else 8
        return {"bytes": 5 * n * (levels * size * (8 * 4 + 6) + 8 * 8),
                "flops": 5 * n * levels * 9 * 30}
    if kind == "elasticity_cg":
        steps = (3 if case["chebyshev"] else 14) * max(_cells(case))
        applications = 5 if case["chebyshev"] else 1
        return {"bytes": 3 * 8 * n * steps * (8 + 4 * (applications - 1)),
                "flops": 330 * n * steps * applications}
    if kind == "adjoint":
        return {"bytes": 40 * n * case["steps"], "flops": 70 * n * case["steps"]}
    return {"bytes": 8 * n * 3 * (10 * 8 + 4) * case["steps"],
            "flops": 30 * n * 3 * 10 * case["steps"]}


def tolerance(case):
    """About four times what `exact`, which sums in another order, shows over the listed and
    drawn cases: rounding for the explicit models, the operators and the gradients (FP32
    arithmetic: its rounding, which the Laplacian in mu amplifies), and for the solves what is
    left at their stopping tolerance."""
    kind, single = case["kind"], case.get("single", False)
    if kind == "precipitate":
        return {"rel": 2e-6 if single else 1e-14}
    if kind == "poisson_apply":
        return {"rel": 2e-6 if single else 1e-14}
    if kind == "adjoint":
        return {"rel": 5e-7 if single else 1e-13}
    return {"ac2d": {"rel": 1e-14}, "ch3d": {"rel": 5e-13}, "elasticity_apply": {"rel": 1e-14},
            "poisson_gmg": {"rel": 5e-8}, "elasticity_cg": {"rel": 1e-7},
            "ac2d_implicit": {"rel": 2e-8}}[kind]


# -------------------------------------------------------------------------- in plain FP64
def _precipitate_mu(c, eta, lat):
    h = eta ** 3 * (6.0 * eta ** 2 - 15.0 * eta + 10.0)
    return 2.0 * (c - 0.1) * (1.0 - h) + 2.0 * (c - 0.9) * h + lat.lap(c)


def _interior(u):
    for d in range(u.dim()):
        u = u.narrow(d, 1, u.shape[d] - 2)
    return u


def _boundary_zero(u):
    out = torch.zeros_like(u)
    _interior(out).copy_(_interior(u))
    return out


def _modes(lat, interior):
    """Per axis (Q, eigenvalues, sqrt(m)) of S = M^{1/2} L M^{-1/2} = Q diag Q^T."""
    modes = []
    for ax in lat.axes:
        m, dense = ax.mass, ax.dense()
        if interior:
            m, dense = m[1:-1], dense[1:-1, 1:-1]
        root = torch.sqrt(m)
        s = root[:, None] * dense / root[None, :]
        values, q = torch.linalg.eigh((0.5 * (s + s.T)).cpu())
        modes.append((q.to(m.device), values.to(m.device), root))
    return modes


def _spectral(u, lat, modes, function):
    """function(L) u by fast diagonalization."""
    for d, (q, _, root) in enumerate(modes):
        t = lat.dim - 1 - d
        u = torch.tensordot(u * lat._along(root, d), q, dims=([t], [0])).movedim(-1, t).contiguous()
    values = sum(lat._along(v, d) for d, (_, v, _) in enumerate(modes))
    u = u * function(values)
    for d, (q, _, root) in enumerate(modes):
        t = lat.dim - 1 - d
        u = torch.tensordot(u, q, dims=([t], [1])).movedim(-1, t).contiguous() / lat._along(root, d)
    return u


class _Elasticity:
    """The linear elasticity operator of the Q2 mesh, assembled cell by cell."""

    def __init__(self, case, given, device):
        self.cells = _cells(case)
        self.mu = given["E"] / (2.0 * (1.0 + given["nu"]))
        self.la = given["E"] * given["nu"] / ((1.0 + given["nu"]) * (1.0 - 2.0 * given["nu"]))
        self.D = torch.tensor([[-3.0, 4.0, -1.0], [-1.0, 0.0, 1.0], [1.0, -4.0, 3.0]],
                              dtype=torch.float64, device=device) / SPACING
        w = torch.tensor([1.0, 4.0, 1.0], dtype=torch.float64, device=device) / 6.0 * SPACING
        self.w = w[:, None, None] * w[None, :, None] * w[None, None, :]
        shape = _shape(case)
        # Dirichlet on every face except y = 0 and z = 0
        self.free = torch.ones(shape, dtype=torch.float64, device=device)
        self.free[:, :, 0] = 0.0
        self.free[:, :, -1] = 0.0
        self.free[:, -1, :] = 0.0
        self.free[-1, :, :] = 0.0

    def _derive(self, v, d):
        # v: (cells z, y, x, kz, ky, kx); derivative along axis d (x = 0) at the nodes
        return torch.tensordot(v, self.D, dims=([5 - d], [1])).movedim(-1, 5 - d)

    def _derive_t(self, v, d):
        return torch.tensordot(v, self.D, dims=([5 - d], [0])).movedim(-1, 5 - d)

    def apply(self, u, plain=False):
        out = torch.zeros_like(u)
        nx, ny, nz = self.cells
        layers = max(1, 100000 // (nx * ny))
        for z0 in range(0, nz, layers):
            z1 = min(nz, z0 + layers)
            part = u[:, 2 * z0:2 * z1 + 1]
            if not plain:
                part = part * self.free[2 * z0:2 * z1 + 1]
            g = [[self._derive(part[c].unfold(0, 3, 2).unfold(1, 3, 2).unfold(2, 3, 2), d)
                  for d in range(3)] for c in range(3)]
            trace = self.la * (g[0][0] + g[1][1] + g[2][2])
            for c in range(3):
                acc = 0.0
                for d in range(3):
                    s = self.mu * (g[c][d] + g[d][c]) + (trace if c == d else 0.0)
                    acc = acc + self._derive_t(self.w * s, d)
                for kz in range(3):
                    for ky in range(3):
                        for kx in range(3):
                            out[c, 2 * z0 + kz:2 * z1 - 1 + kz:2, ky:ky + 2 * ny - 1:2,
                                kx:kx + 2 * nx - 1:2] += acc[:, :, :, kz, ky, kx]
        return out * self.free


def _exact_elasticity_cg(case, given, device):
    op = _Elasticity(case, given, device)
    lat = _Lattice(case, device)
    root = 1.0 / torch.sqrt(lat.mass())
    lift = torch.zeros((3,) + _shape(case), dtype=torch.float64, device=device)
    lift[0, :, :, 0] = -1.0
    diagonal = root * root  # equilibrates the rows of edge, face and cell nodes
    r = -op.apply(lift, plain=True)
    x = torch.zeros_like(r)
    z = diagonal * r
    p, rz = z.clone(), torch.sum(r * z)
    goal = 1e-13 * math.sqrt(float(rz))
    for _ in range(8000):
        ap = op.apply(p)
        alpha = rz / torch.sum(p * ap)
        x += alpha * p
        r -= alpha * ap
        z = diagonal * r
        new = torch.sum(r * z)
        if math.sqrt(float(new)) <= goal:
            break
        p = z + (new / rz) * p
        rz = new
    return [x[c] + lift[c] for c in range(3)]


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    given, kind = _inputs(case, seed, device), case["kind"]
    if kind in ("elasticity_apply", "elasticity_cg"):
        if kind == "elasticity_cg":
            return _exact_elasticity_cg(case, given, device)
        u, op = given["u"], _Elasticity(case, given, device)
        for _ in range(APPLICATIONS):
            u = op.apply(u)
        return u
    lat = _Lattice(case, device)
    if kind == "ac2d":
        phi = given["phi"]
        for _ in range(case["steps"]):
            phi = phi - DT_AC2D * (phi ** 3 - phi) - DT_AC2D * 1.5 * lat.lap(phi)
        return {"phi": phi}
    if kind == "ch3d":
        c, mu = given["c"], given["mu"]
        for _ in range(case["steps"]):
            c = c - DT_CH * lat.lap(mu)
            mu = 2.0 * c * (1.0 - c) * (1.0 - 2.0 * c) + lat.lap(c)
        return {"c": c, "mu": mu}
    if kind == "precipitate":
        c, mu, eta, dt = given["c"], given["mu"], given["eta"], DT_PRECIPITATE
        for _ in range(case["steps"]):
            slope = 30.0 * eta ** 2 * (1.0 - eta) ** 2
            force = (((c - 0.9) ** 2 - (c - 0.1) ** 2) * slope +
                     2.0 * eta * (1.0 - eta) * (1.0 - 2.0 * eta))
            eta = eta - dt * force - dt * lat.lap(eta)
            c = c - dt * lat.lap(mu)
            mu = _precipitate_mu(c, eta, lat)
        return {"c": c, "mu": mu, "eta": eta}
    if kind == "poisson_apply":
        u, mass = given["u"].double(), lat.mass()
        for _ in range(APPLICATIONS):
            u = _boundary_zero(mass * lat.lap(_boundary_zero(u)))
        return u
    if kind == "poisson_gmg":
        out = torch.zeros_like(given["f"])
        inner = _spectral(_interior(given["f"]).contiguous(), lat, _modes(lat, True), lambda v: 1.0 / v)
        _interior(out).copy_(inner)
        return out
    if kind == "adjoint":
        phi, lam, mass, dt = given["phi"], given["lam"], lat.mass(), DT_ADJOINT
        history = []
        for _ in range(case["steps"]):
            history.append(phi)
            phi = phi - dt * (phi ** 3 - phi) - dt * 1.5 * lat.lap(phi)
        dL = dkappa = 0.0
        for p in reversed(history):
            lap = lat.lap(p)
            dL += float(torch.sum(lam * (-dt * (p ** 3 - p) - dt * 1.5 * lap)))
            dkappa += float(torch.sum(lam * (-dt * lap)))
            lam = lam - dt * (3.0 * p * p - 1.0) * lam - dt * 1.5 * mass * lat.lap(lam / mass)
        return {"dL": dL, "dkappa": dkappa, "dphi0": lam}
    # implicit Allen-Cahn: (1 + dt kappa L) n = n_old - dt f'(n), a contraction at this dt
    old, dt, modes = given["n"], DT_IMPLICIT, _modes(lat, False)
    for _ in range(case["steps"]):
        n = old
        for _ in range(100):
            new = _spectral(old - dt * 4.0 * n * (n - 1.0) * (n - 0.5), lat, modes,
                            lambda v: 1.0 / (1.0 + dt * 2.0 * v))
            change = float((new - n).abs().max())
            n = new
            if change < 1e-15:
                break
        old = n
    return {"n": n}
