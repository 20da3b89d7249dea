"""stencil_column_kernel (small lattices) against the tiled kernel on the same operators.

Lattices: 2 cells per axis (every neighbour wraps or reflects), planes of just under, at and
over a multiple of 256 nodes (a workgroup), 1 to 3 planes beyond a multiple of 4 (a thread's
planes), 2-D.  Operators with and without Dirichlet faces, one and no stencil operand, value
inputs that alias the operand, Q1 and Q2, FP64, FP32, and FP32 arithmetic on the FP64 state.

Tolerance: both kernels form the same sums in the same order; only the compiler's contraction
of the hook's products may differ, one rounding of terms no larger than the largest output:
8 eps (FP64: 2e-15, FP32: 1e-6).
"""

import numpy as np
import pytest

from phasefield_amd import Context, prm
from phasefield_amd.capi import (AGE_LATEST, FP32, FP64, OP_LHS, OP_RHS, SCALE_INVM,
                                 SCALE_INVM_SQRT, SCALE_NONE)
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu

TOL = {FP64: 2e-15, FP32: 1e-6}
# 256 nodes: 16 x 16 (periodic Q1), 8 x 8 cells (periodic Q2); 289 and 285: over and under
MESHES = {"smallest": (2, 2, 2), "block": (16, 16, 9), "under": (5, 51, 6), "over": (17, 17, 7),
          "thin": (3, 40, 2)}


def pair(app, text):
    tile, column = Context(app, text), Context(app, text)
    tile.set_option("stencil_min_nodes", 0)
    column.set_option("stencil_min_nodes", 10 ** 12)
    return tile, column


def compare(ctxs, torch, block, which, scaling, precision, src=None):
    outs = []
    dtype = torch.float64 if precision == FP64 else torch.float32
    for ctx in ctxs:
        dst = torch.full((ctx.info.n_nodes,), 3.0, dtype=dtype, device="cuda")
        s = src.to(dtype) if src is not None else None
        for _ in range(2):  # the first application compares the paths itself
            ctx.apply_operator(block, which, scaling, precision, s.data_ptr() if src is not None else 0,
                               dst.data_ptr())
        torch.cuda.synchronize()
        outs.append(dst.double().cpu().numpy())
    assert rel_err(outs[1], outs[0]) <= TOL[precision], (block, which, scaling, precision)


@pytest.mark.parametrize("mesh", list(MESHES))
@pytest.mark.parametrize("model", ["cahn_hilliard", "precipitate", "allen_cahn_2d"])
def test_column_matches_tile_on_explicit_blocks(device, model, mesh):
    import torch

    cells = list(MESHES[mesh])
    if model == "cahn_hilliard":
        app, text = "cahn_hilliard_3d_q2", prm.cahn_hilliard(refinement=0, subdivisions=cells)
        blocks, n = (0, 1), 2
    elif model == "precipitate":
        app = "precipitate_3d_q1"
        text, blocks, n = prm.precipitate(refinement=0, subdivisions=cells), (0, 1, 2), 3
    else:
        app, blocks, n = "allen_cahn_2d_q1", (1,), 1
        text = prm.allen_cahn(dim=2, refinement=0, subdivisions=cells[:2])
    ctxs = pair(app, text)
    rng = np.random.default_rng(5)
    for f in range(n):
        values = rng.uniform(0.1, 0.9, ctxs[0].full_shape())
        for ctx in ctxs:
            for age in (0, 1):
                ctx.set_field(f, values, age)
    for block in blocks:
        for scaling in (SCALE_INVM, SCALE_NONE, SCALE_INVM_SQRT):
            compare(ctxs, torch, block, OP_RHS, scaling, FP64)
        compare(ctxs, torch, block, OP_RHS, SCALE_INVM, FP32)
    # increments, the NaN probe included, in both precisions of the explicit update
    for precision in ("double", "single"):
        for ctx in ctxs:
            ctx.set_option("explicit_precision", precision)
            ctx.set_time(1, 1e-3)
            assert ctx.run(4) == 0
        for f in range(n):
            a, b = (ctx.get_field(f, AGE_LATEST) for ctx in ctxs)
            assert rel_err(b, a) <= (1e-14 if precision == "double" else 1e-5)


@pytest.mark.parametrize("mesh", list(MESHES))
@pytest.mark.parametrize("dim", [2, 3])
def test_column_matches_tile_on_dirichlet_lhs(device, dim, mesh):
    import torch

    text = prm.poisson(dim=dim, refinement=0, subdivisions=list(MESHES[mesh])[:dim], mg_depth=1,
                       preconditioner="None")
    ctxs = pair(f"poisson_{dim}d_q2", text)
    rng = np.random.default_rng(6)
    src = torch.tensor(rng.uniform(-1.0, 1.0, ctxs[0].info.n_nodes), device=device)
    for precision in (FP64, FP32):
        for scaling in (SCALE_NONE, SCALE_INVM_SQRT):
            compare(ctxs, torch, 1, OP_LHS, scaling, precision, src)
    # a right-hand side without a stencil operand
    values = rng.uniform(-1.0, 1.0, ctxs[0].full_shape())
    for ctx in ctxs:
        ctx.set_field(1, values, 0)
    compare(ctxs, torch, 1, OP_RHS, SCALE_NONE, FP64)
