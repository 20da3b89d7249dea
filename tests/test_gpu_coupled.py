"""The coupled stencil of a 3-D vector field (linear elasticity) against the generic cell
kernel: same operator, another order of the sums.

Meshes: the smallest lattice the stencil takes (5 nodes per axis), one below it (generic path),
tile widths of 32 to 64 columns and their remainders, row-pair and z-chunk remainders, periodic
axes, unequal spacings.  Boundaries: none, some and all faces Dirichlet, so that the boundary
terms of natural faces, their edges and corners are all summed.

Tolerance: an output is a sum of about 100 products; in another order it moves by at most
100 eps times the sum of their magnitudes, which is within 10 of the largest output:
1e3 * 1.1e-16 ~ 1e-13 (FP64) and 1e3 * 6e-8 ~ 6e-5 (FP32).
"""

import numpy as np
import pytest

from phasefield_amd import Context, prm
from phasefield_amd.capi import (FP32, FP64, OP_LHS, OP_LHS_PLAIN, SCALE_INVM, SCALE_INVM_SQRT,
                                 SCALE_NONE)
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu

APP = "mechanics_3d_q2"
MIXED = ("Dirichlet", "Dirichlet", "Natural", "Dirichlet", "Natural", "Dirichlet")
NATURAL = ("Natural",) * 6
# cells, periodic axes, conditions
MESHES = {
    "smallest": ((2, 2, 2), "", NATURAL),
    "one_cell": ((1, 3, 2), "", MIXED),
    "reference_faces": ((7, 5, 6), "", MIXED),
    "natural": ((4, 9, 3), "", NATURAL),
    "all_dirichlet": ((5, 4, 7), "", ("Dirichlet",) * 6),
    "tile_31_32": ((31, 3, 2), "", ("Natural", "Dirichlet", "Natural", "Natural", "Dirichlet",
                                    "Natural")),
    "tile_33": ((33, 8, 3), "", MIXED),
    "wide": ((65, 4, 2), "", NATURAL),
    "tall": ((3, 40, 4), "", NATURAL),
    "deep": ((4, 3, 41), "", MIXED),
    "periodic_x": ((16, 5, 4), "x", NATURAL),
    "periodic_yz": ((6, 17, 9), "yz", ("Dirichlet",) + ("Natural",) * 5),
    "periodic": ((32, 6, 5), "xyz", NATURAL),
}


def mesh_text(cells, periodic, conditions):
    out = []
    for line in prm.mechanics(refinement=0, conditions=conditions).splitlines():
        w = line.split()
        if len(w) > 3 and w[0] == "set" and w[1] in ("x", "y", "z"):
            d = "xyz".index(w[1])
            if w[2] == "size":
                line = f"  set {w[1]} size = {cells[d] * (1.0 + 0.25 * d)!r}"
            elif w[2] == "subdivisions":
                line = f"  set {w[1]} subdivisions = {cells[d]}"
            elif w[2] == "periodic":
                line = f"  set {w[1]} periodic = {'true' if w[1] in periodic else 'false'}"
        out.append(line)
    return "\n".join(out) + "\n"


def apply(ctx, torch, src, which, scaling, precision):
    dst = torch.full_like(src, 7.0)
    ctx.apply_operator(1, which, scaling, precision, src.data_ptr(), dst.data_ptr())
    torch.cuda.synchronize()
    return dst.cpu().numpy()


@pytest.mark.parametrize("mesh", list(MESHES))
def test_coupled_stencil_matches_generic(device, mesh):
    import torch

    cells, periodic, conditions = MESHES[mesh]
    text = mesh_text(cells, periodic, conditions)
    fast, slow = Context(APP, text), Context(APP, text)
    slow.set_option("operator_path", "generic")
    rng = np.random.default_rng(11)
    src = torch.tensor(rng.uniform(-1.0, 1.0, 3 * fast.info.n_nodes), device=device)
    for which in (OP_LHS, OP_LHS_PLAIN):
        for scaling in (SCALE_NONE, SCALE_INVM, SCALE_INVM_SQRT):
            for _ in range(2):  # the first application compares the paths itself
                got = apply(fast, torch, src, which, scaling, FP64)
            ref = apply(slow, torch, src, which, scaling, FP64)
            assert rel_err(got, ref) <= 1e-13, (mesh, which, scaling, rel_err(got, ref))
    for _ in range(2):
        got = apply(fast, torch, src.float(), OP_LHS, SCALE_NONE, FP32)
    ref = apply(slow, torch, src, OP_LHS, SCALE_NONE, FP64)
    assert rel_err(got, ref) <= 6e-5, (mesh, rel_err(got, ref))
    taken = "solve block 1 (lhs): coupled stencil\n" in fast.output_log()
    assert taken == all(n >= 5 for n in fast.info.nodes), fast.output_log()
    # inverse diagonal: from the coefficients (fast) and probed cell by cell (slow)
    a, b = torch.empty_like(src), torch.empty_like(src)
    fast.inverse_diagonal(1, SCALE_INVM_SQRT, FP64, a.data_ptr())
    slow.inverse_diagonal(1, SCALE_INVM_SQRT, FP64, b.data_ptr())
    err = float(((a - b).abs() / b.abs()).max())
    assert err <= 1e-13, (mesh, err)


def fresh_pair(cells, device, torch):
    """A fresh context, one on the generic path, and a random block vector."""
    text = mesh_text(cells, "", MIXED)
    fast, slow = Context(APP, text), Context(APP, text)
    slow.set_option("operator_path", "generic")
    src = torch.tensor(np.random.default_rng(12).uniform(-1.0, 1.0, 3 * fast.info.n_nodes),
                       device=device)
    return fast, slow, src


def test_first_application_can_be_captured(device):
    """Nothing can be compared under capture: the generic kernel is recorded, and replays give
    its bits whatever path eager applications in between take."""
    import torch

    fast, slow, src = fresh_pair((6, 5, 4), device, torch)
    fast.set_option("synchronize", 0)
    dst = torch.zeros_like(src)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(fast.stream()),
                          capture_error_mode="relaxed"):
        fast.apply_operator(1, OP_LHS, SCALE_NONE, FP64, src.data_ptr(), dst.data_ptr())
    for replay in range(4):
        src.uniform_(-1.0, 1.0)
        dst.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ref = apply(slow, torch, src, OP_LHS, SCALE_NONE, FP64)
        assert np.array_equal(dst.cpu().numpy(), ref), replay
        assert rel_err(apply(fast, torch, src, OP_LHS, SCALE_NONE, FP64), ref) <= 1e-13
    assert "coupled stencil" in fast.output_log()


def test_scratch_too_small_to_compare(device):
    """142 x 142 x 142 nodes and more: the reference of the comparison does not fit the 64 MiB
    of scratch, so an application without allocation runs the generic kernel until one with
    allocation has checked the plan."""
    import torch

    fast, slow, src = fresh_pair((71, 71, 71), device, torch)
    dst, ref = torch.empty_like(src), torch.empty_like(src)
    args = (1, OP_LHS, SCALE_NONE, FP64, src.data_ptr())
    slow.apply_operator(*args, ref.data_ptr())
    fast.apply_operator_noalloc(*args, dst.data_ptr())
    torch.cuda.synchronize()
    assert torch.equal(dst, ref) and "coupled stencil" not in fast.output_log()
    fast.apply_operator(*args, dst.data_ptr())
    assert "coupled stencil" in fast.output_log()
    again = torch.empty_like(dst)
    fast.apply_operator_noalloc(*args, again.data_ptr())
    torch.cuda.synchronize()
    assert torch.equal(dst, again)
    assert rel_err(dst.cpu().numpy(), ref.cpu().numpy()) <= 1e-13


def test_small_scratch_compares(device):
    """129 x 129 x 129 nodes: the reference fits, and the first application without
    allocation checks the plan."""
    import torch

    fast, slow, src = fresh_pair((64, 64, 64), device, torch)
    dst, ref = torch.empty_like(src), torch.empty_like(src)
    args = (1, OP_LHS, SCALE_NONE, FP64, src.data_ptr())
    slow.apply_operator(*args, ref.data_ptr())
    fast.apply_operator_noalloc(*args, dst.data_ptr())
    torch.cuda.synchronize()
    assert "coupled stencil" in fast.output_log()
    assert rel_err(dst.cpu().numpy(), ref.cpu().numpy()) <= 1e-13


@pytest.mark.parametrize("zeros, until", [(1, 1), (2, 3), (5, 7), (9, 3)])
def test_zero_operand_checks_nothing(device, zeros, until):
    """An application to zero agrees whatever the coefficients are: the inverse diagonal is
    probed on the generic path (its bits) until an application to something has been compared,
    the next one after one application to zero, at the latest the `until`-th after more."""
    import torch

    fast, slow, src = fresh_pair((6, 5, 4), device, torch)
    diag, ref = torch.empty_like(src), torch.empty_like(src)
    slow.inverse_diagonal(1, SCALE_INVM_SQRT, FP64, ref.data_ptr())
    generic = apply(slow, torch, src, OP_LHS, SCALE_NONE, FP64)
    for _ in range(zeros):
        assert not apply(fast, torch, torch.zeros_like(src), OP_LHS, SCALE_NONE, FP64).any()
        fast.inverse_diagonal(1, SCALE_INVM_SQRT, FP64, diag.data_ptr())
        assert torch.equal(diag, ref)
    for k in range(until):
        fast.inverse_diagonal(1, SCALE_INVM_SQRT, FP64, diag.data_ptr())
        assert torch.equal(diag, ref)
        got = apply(fast, torch, src, OP_LHS, SCALE_NONE, FP64)
        assert np.array_equal(got, generic) == (k < until - 1)
        assert rel_err(got, generic) <= 1e-13
    fast.inverse_diagonal(1, SCALE_INVM_SQRT, FP64, diag.data_ptr())
    assert not torch.equal(diag, ref)  # from the coefficients
    assert float(((diag - ref).abs() / ref.abs()).max()) <= 1e-13
