"""Routing of equation hooks between the split (stencil) path and the generic cell path
is safe for hooks whose flux coefficients branch (application switching_2d_q2):

* block 1, coefficient switching at c > 1: the structure probe (random states with
  values up to +-50) sees a non-constant coefficient and routes it to the generic path;
* block 2, coefficient switching at increment 3: the probe sees the dependence on the
  increment and re-derives the plan whenever the increment changes;
* block 3, coefficient switching at c > 60 (beyond the probe's values): the comparison
  with the generic path at the plan's first use on the real fields (c reaches 70)
  drops the split plan and says so in the output log;
* block 4, the same coefficient in the lhs of a linear solve.

Every field matches the oracle (which evaluates every hook at every quadrature point)
after 6 increments, across the switch at increment 3.
"""

from __future__ import annotations

import numpy as np
import pytest

from phasefield_amd import Context, PPFError, prm
from phasefield_amd.capi import AGE_LATEST
from oracle.binding import Oracle
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu

APP = "switching_2d_q2"


def test_branching_hooks_match_oracle(device):
    text = prm.switching(steps=6)
    ctx, orc = Context(APP, text), Oracle(APP, text)
    assert ctx.run(6) == 0 and orc.run(6) == 0
    for f in range(4):
        err = rel_err(ctx.get_field(f, AGE_LATEST).ravel(), orc.get_field(f, AGE_LATEST))
        print(f"field {f}: relative difference from the oracle {err:.2e}", flush=True)
        assert err <= 1e-10, (f, err)
    log = ctx.output_log()
    print(log, flush=True)
    assert "solve block 3 (rhs): the split operator differs from the generic path" in log
    assert "solve block 1 " not in log and "solve block 0 " not in log


def test_forced_split_path_refuses_value_branch(device):
    ctx = Context(APP, prm.switching(steps=2))
    ctx.set_option("operator_path", "split")
    with pytest.raises(PPFError) as e:
        ctx.run(2)
    assert "does not qualify" in str(e.value)


@pytest.mark.parametrize("preconditioner", ["None", "Chebyshev"])
def test_plan_dropped_by_a_solve(device, preconditioner):
    """Block 4 (linear), the same branch in its lhs: the first solve drops the plan on its
    right-hand side (its own first applications, to zero, agree on anything), and every step
    runs the generic path.

    Tolerance: residuals of 1e-10 on an operator whose smallest eigenvalue in M^-1/2 scaling is
    1 (its value term); 1e-8 leaves the rounding of about 100 steps."""
    text = prm.switching(steps=3, preconditioner=preconditioner)
    ctx, orc = Context(APP, text), Oracle(APP, text)
    assert ctx.run(3) == 0 and orc.run(3) == 0
    assert "solve block 4 (lhs): the split operator differs from the generic path" in ctx.output_log()
    assert rel_err(ctx.get_field(4, AGE_LATEST).ravel(), orc.get_field(4, AGE_LATEST)) <= 1e-8
    values = np.random.default_rng(8).uniform(-10.0, 70.0, ctx.full_shape())
    for c in (ctx, orc):
        c.set_field(0, values, 0)
    st, ref = ctx.linear_solve(4), orc.linear_solve(4)
    assert st.converged and st.iterations == ref["iterations"] > 10
    assert rel_err(ctx.get_field(4, AGE_LATEST).ravel(), orc.get_field(4, AGE_LATEST)) <= 1e-8
