"""The Allen-Cahn forward and adjoint kernels at the edges of their plane groups (4 planes per
thread) and workgroups (256 nodes of the x-y plane), against the oracle.

Meshes of 1 to 9 planes beyond the smallest, planes of under, exactly and over 256 nodes,
periodic and natural boundaries.

Tolerance: a step is a sum of about 20 products of values of order one, repeated 7 times:
7 * 20 * 1.1e-16 ~ 2e-14, and the sums dL, dkappa add rounding over the nodes -> 1e-12.
"""

import numpy as np
import pytest

from oracle.binding import Oracle
from phasefield_amd import Context, prm
from phasefield_amd.capi import FP64
from tests.helpers import rel_err, to_full, to_stored

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("cells", [(4, 4, 2), (5, 7, 3), (16, 16, 4), (6, 2, 5), (18, 16, 6),
                                   (14, 18, 10), (15, 17, 7), (4, 4, 8), (3, 90, 9)])
def test_adjoint_matches_oracle(device, oracle_libs, cells, periodic):
    import torch

    if periodic and any(c % 2 for c in cells):
        cells = tuple(c + c % 2 for c in cells)  # the oracle's periodic meshes have even counts
    text = prm.allen_cahn(dim=3, refinement=0, subdivisions=list(cells), steps=7, dt=0.02)
    lines = []
    for line in text.splitlines():
        w = line.split()
        if len(w) > 3 and w[2] == "size":
            line = f"  set {w[1]} size = {float(cells['xyz'.index(w[1])])!r}"
        elif len(w) > 3 and w[2] == "periodic" and not periodic:
            line = f"  set {w[1]} periodic = false"
        lines.append(line)
    text = "\n".join(lines) + "\n"
    ctx, orc = Context("allen_cahn_3d_q1", text), Oracle("allen_cahn_3d_q1", text)
    info, n, every = ctx.info, 7, 3
    rng = np.random.default_rng(8)
    phi = to_full(to_stored(rng.uniform(-1.0, 1.0, ctx.full_shape()), info), info)
    lam = to_full(to_stored(rng.uniform(-1.0, 1.0, ctx.full_shape()), info), info)
    lam[orc.lumped_mass() == 0] = 0.0  # image entries: the oracle folds them onto masters
    d_phi = torch.tensor(to_stored(phi, info), device=device)
    d_lam = torch.tensor(to_stored(lam, info), device=device)
    out, grad = torch.empty_like(d_phi), torch.empty_like(d_phi)
    ctx.adjoint_forward(d_phi.data_ptr(), 1.0, 1.5, n, FP64, out.data_ptr())
    dL, dk = ctx.adjoint_vjp(d_phi.data_ptr(), d_lam.data_ptr(), 1.0, 1.5, n, every, FP64,
                             grad.data_ptr())
    assert rel_err(to_full(out.cpu().numpy(), info), orc.adjoint_forward(phi, 1.0, 1.5, n)) <= 1e-12
    oL, ok, og = orc.adjoint_vjp(phi, lam, 1.0, 1.5, n)
    assert rel_err(grad.cpu().numpy(), to_stored(og, info)) <= 1e-12
    scale = np.abs(lam).sum()
    assert abs(dL - oL) <= 1e-12 * (abs(oL) + 1e-2 * scale)
    assert abs(dk - ok) <= 1e-12 * (abs(ok) + 1e-2 * scale)
