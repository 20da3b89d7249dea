"""CG steps enqueued ahead of the residual the host reads: the step count, the residual and the
iterate must be those of a loop that looks at every residual before the next step.

Cases: vectors of one workgroup, of several partial sums and of more than one per thread
(125, 2 197, 35 937 and 274 625 nodes), stopped by the tolerance, by an iteration limit of 1,
2 and 7 (the limit falls before and after steps enqueued ahead), and by an initial residual
below the tolerance; each against the oracle's CG.

Tolerance: n steps of CG in FP64 with other summation orders; rounding grows with the steps
and with the condition number (at most 2e4 here): 100 steps * 2e4 * 1.1e-16 ~ 2e-10 -> 1e-9.
"""

import pytest

from oracle.binding import Oracle
from phasefield_amd import Context, prm
from phasefield_amd.capi import AGE_LATEST
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("refinement, limit", [(1, 1000), (1, 1), (2, 2), (2, 1000), (3, 7),
                                               (4, 1000), (5, 7)])
@pytest.mark.parametrize("preconditioner", ["None", "Chebyshev"])
def test_cg_stops_like_the_oracle(device, oracle_libs, refinement, limit, preconditioner):
    size = {1: 2, 2: 6, 3: 8, 4: 16, 5: 32}[refinement]
    text = prm.poisson(dim=3, refinement=0, subdivisions=[size] * 3, mg_depth=1, tolerance=1e-9,
                       preconditioner=preconditioner, max_iterations=limit)
    ctx, orc = Context("poisson_3d_q2", text), Oracle("poisson_3d_q2", text)
    for c in (ctx, orc):
        c.solve_block(0)
        c.set_time(1, 0.0)
    st, ref = ctx.linear_solve(1), orc.linear_solve(1)
    assert st.iterations == ref["iterations"] and bool(st.converged) == bool(ref["converged"])
    assert (st.iterations == limit) == (limit < 1000)
    assert rel_err(ctx.get_field(0, AGE_LATEST).ravel(), orc.get_field(0, AGE_LATEST)) <= 1e-9
    # again from the solution: no step if it converged, `limit` more otherwise
    st, ref = ctx.linear_solve(1), orc.linear_solve(1)
    assert st.iterations == ref["iterations"]
    assert rel_err(ctx.get_field(0, AGE_LATEST).ravel(), orc.get_field(0, AGE_LATEST)) <= 1e-9


@pytest.mark.parametrize("cells, workgroups", [((255, 256), 1024), ((256, 256), 1029),
                                               ((300, 300), 1411)])
def test_cg_around_the_limit_of_partial_sums(device, oracle_libs, cells, workgroups):
    """2-D lattices of the column kernel on both sides of 1024 workgroups, the partial sums that
    d.Ad of the operator's own launch has room for: 511 x 513, 513 x 513 and 601 x 601 nodes.
    The solve is cut short: the iterates of 25 steps are compared (condition number 1e5)."""
    text = prm.poisson(dim=2, refinement=0, subdivisions=list(cells), mg_depth=1, tolerance=1e-9,
                       preconditioner="None", max_iterations=25)
    ctx, orc = Context("poisson_2d_q2", text), Oracle("poisson_2d_q2", text)
    assert (ctx.info.n_nodes + 255) // 256 == workgroups
    for c in (ctx, orc):
        c.solve_block(0)
        c.set_time(1, 0.0)
    for _ in range(2):  # from zero, then on from there
        st, ref = ctx.linear_solve(1), orc.linear_solve(1)
        assert st.iterations == ref["iterations"] == 25
        assert rel_err(ctx.get_field(0, AGE_LATEST).ravel(), orc.get_field(0, AGE_LATEST)) <= 1e-9
