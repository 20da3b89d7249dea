"""Order of the tiled kernel's workgroups (stencil_map): bands of tile rows per XCD against the
linear order, bit for bit (the same tiles, each computed alone).

Tile rows (8 lattice rows each): 1 and 3 (XCDs without a band), 9 and 11 (a short last band and
XCDs without one), 16 (even).  Lattices end in partial tiles along y, in columns beyond the last
whole tile along x and in a partial z chunk; Cahn-Hilliard increments (periodic, NaN probe on
the launch) and the Dirichlet Poisson operator in FP64 and FP32.
"""

import numpy as np
import pytest

from phasefield_amd import Context, prm
from phasefield_amd.capi import AGE_LATEST, FP32, FP64, OP_LHS, SCALE_NONE

pytestmark = pytest.mark.gpu


def contexts(app, text):
    out = []
    for order in ("linear", "band"):
        ctx = Context(app, text)
        ctx.set_option("stencil_min_nodes", 0)
        ctx.set_option("stencil_map", order)
        out.append(ctx)
    return out


@pytest.mark.parametrize("rows", [4, 11, 33, 43, 64])
def test_bands_match_the_linear_order(device, rows):
    import torch

    text = prm.cahn_hilliard(refinement=0, subdivisions=[33, rows, 7])
    ctxs = contexts("cahn_hilliard_3d_q2", text)
    for ctx in ctxs:
        assert ctx.run(4) == 0
    for f in range(2):
        a, b = (ctx.get_field(f, AGE_LATEST) for ctx in ctxs)
        assert np.isfinite(a).all() and np.array_equal(a, b), f

    text = prm.poisson(dim=3, refinement=0, subdivisions=[35, rows, 5], mg_depth=1,
                       preconditioner="None")
    ctxs = contexts("poisson_3d_q2", text)
    src = torch.tensor(np.random.default_rng(4).uniform(-1.0, 1.0, ctxs[0].info.n_nodes),
                       device=device)
    for precision, dtype in ((FP64, torch.float64), (FP32, torch.float32)):
        s = src.to(dtype)
        outs = [torch.full_like(s, 5.0) for _ in ctxs]
        for ctx, dst in zip(ctxs, outs):
            for _ in range(2):  # the first application compares the paths itself
                ctx.apply_operator(1, OP_LHS, SCALE_NONE, precision, s.data_ptr(), dst.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(*outs), precision
