"""V-cycles with smoother steps fused into the operator and one-launch transfers against the
oracle: equal CG counts and solutions.

Smoother degrees 1 to 5 (the iterate changes buffers in every fused step; odd counts start
elsewhere), lattices on both sides of the fusing limit, ragged coarse meshes (transfer columns
and plane groups with remainders), 2-D and 3-D, Q2 (Poisson, all faces Dirichlet) and Q1
(implicit Allen-Cahn, natural and periodic boundaries), FP64 and FP32 levels.

Tolerance: both solve to 1e-10 of the initial residual in the same number of CG steps; the
solutions then differ by that times the condition number of the preconditioned system (about
1): 1e-8 leaves room for it.
"""

import numpy as np
import pytest

from oracle.binding import Oracle
from phasefield_amd import Context, prm
from phasefield_amd.capi import AGE_LATEST
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("min_nodes", [0, 10 ** 12])
@pytest.mark.parametrize("dim, cells, refinement, degree", [
    (3, (1, 1, 1), 3, 4), (3, (2, 1, 3), 2, 3), (3, (1, 3, 1), 3, 1), (3, (3, 2, 1), 2, 5),
    (3, (1, 1, 5), 2, 2), (2, (3, 1), 4, 4), (2, (1, 5), 3, 3), (2, (7, 2), 2, 2),
])
def test_poisson_gmg(device, oracle_libs, dim, cells, refinement, degree, min_nodes):
    text = prm.poisson(dim=dim, refinement=refinement, mg_depth=refinement, tolerance=1e-10,
                       smoother_degree=degree, subdivisions=list(cells))
    app = f"poisson_{dim}d_q2"
    ctx, orc = Context(app, text), Oracle(app, text)
    ctx.set_option("stencil_min_nodes", min_nodes)
    rng = np.random.default_rng(3)
    f = rng.standard_normal(ctx.full_shape())
    for c in (ctx, orc):
        c.set_field(1, f, 0)
        c.set_time(1, 0.0)
    ref = orc.linear_solve(1)
    u = np.array(orc.get_field(0, AGE_LATEST))
    ctx.set_option("linear_initial_guess", "zero")
    for precision in ("double", "single"):
        ctx.set_option("mg_level_precision", precision)
        for _ in range(3):  # eager V-cycles, then captured ones
            st = ctx.linear_solve(1)
            assert st.converged and abs(st.iterations - ref["iterations"]) <= 1
            assert precision == "single" or st.iterations == ref["iterations"]
            assert rel_err(ctx.get_field(0, AGE_LATEST).ravel(), u) <= 1e-8


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("cells, refinement", [((1, 1), 5), ((3, 1), 3), ((2, 5), 2)])
def test_allen_cahn_q1_gmg(device, oracle_libs, cells, refinement, periodic):
    text = prm.allen_cahn_implicit(refinement=refinement, steps=3, dt=0.5, linear_tolerance=1e-12,
                                   newton_tolerance=1e-10, preconditioner="GMG",
                                   mg_depth=min(refinement, 3), subdivisions=list(cells),
                                   periodic=periodic)
    app = "allen_cahn_implicit_2d_q1"
    ctx, orc = Context(app, text), Oracle(app, text)
    for inc in range(3):
        assert ctx.solve_increment() == 0 and orc.solve_increment() == 0
        if inc:
            g, o = ctx.last_newton_stats(1), orc.last_newton_stats(1)
            assert g.iterations == o["iterations"]
            assert abs(g.linear_iterations - o["linear_iterations"]) <= g.iterations
        assert rel_err(ctx.get_field(0, AGE_LATEST).ravel(), orc.get_field(0, AGE_LATEST)) <= 1e-8
