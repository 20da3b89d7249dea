"""Host logic of the runtime on the CPU: small headers of phasefield_amd/csrc compiled into
native programs (no GPU calls)."""

from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

from phasefield_amd.build import HIP_FLAGS, HIPCC

ROOT = Path(__file__).resolve().parent.parent


def native(tmp_path, name, compiler=("g++",)):
    """Compiles tests/native/<name>, runs it and returns its "key: value" lines."""
    exe = tmp_path / Path(name).stem
    subprocess.run([*compiler, "-std=c++20", "-O1", f"-I{ROOT / 'phasefield_amd' / 'include'}",
                    f"-I{ROOT / 'phasefield_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / name), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    return dict(line.split(": ", 1) for line in out.splitlines())


def test_host_scalars_ignore_what_the_memory_held(tmp_path):
    out = native(tmp_path, "host_scalars.cc")
    # no entry counts as sent before its scalar is, also not one with the awaited tag
    assert out["first"] == "1" and out["stale"] == "0" and out["missed"] == "0"
    assert out["last"] == str(2 ** 31 - 1) and out["wrapped"] == "1" and out["empty"] == "0"


@pytest.fixture(scope="module")
def logic(tmp_path_factory):
    """Host evaluations of functions that the kernels and their launches share."""
    return native(tmp_path_factory.mktemp("logic"), "runtime_logic.hip",
                  (HIPCC, *(f for f in HIP_FLAGS if f != "-shared")))


def test_cg_turn_is_uniform_while_it_ends(logic):
    # A launch whose waves find 0 or the launch's own tag, by when they look, must not part:
    # both stay for the barriers of its sums.  Only later launches leave at once.
    assert logic["turn_open"] == "00" and logic["turn_racing"] == "0"
    assert logic["turn_after"] == "1" and logic["turn_last_tag"] == "10"


def test_smoother_step_is_for_its_application_only(tmp_path):
    out = native(tmp_path, "smoother_request.cc")
    assert out["own"] == "10" and out["taken"] == "017"
    for other in ("before", "other_block", "other_dst", "other_src"):
        assert out[other] == "0", other
    # an application that compares A x takes none, and says so to the caller
    assert out["withdrawn"] == "00"
    # nothing is left for the next launch where the application threw or did not take it
    assert out["after_throw"] == "00" and out["not_taken"] == "00"


def test_transfer_launches_check_both_planes(logic):
    # The restriction runs over the coarse plane and reads the fine one with 32-bit indices.
    assert logic["transfer_fits"] == "00"
    assert logic["transfer_fine_plane"] == "1111" and logic["transfer_planes"] == "11"


@pytest.mark.parametrize("degree", [1, 2])
def test_transfers_read_only_what_their_outputs_take(logic, degree):
    # Stray taps (weight zero, at a node the output does not depend on: 0 * NaN would reach
    # it) and positions outside the lattice, of the restriction and of the prolongation.
    assert logic[f"taps_q{degree}"] == "0 0 0 0"


def test_comparison_of_zero_with_zero_decides_nothing(logic):
    # 0 agrees, 1 differs, 2 undecided
    assert logic["check"] == "012111"
    # the next application compares again, then fewer and fewer
    assert logic["check_again"].split() == ["0", "2", "6", "14", "1048574", "1048574"]


def test_comparison_is_kept_by_the_same_path_only(logic):
    assert logic["keeps_check"] == "100" "010" "000"


def test_tile_options_reach_the_tiles(logic):
    assert logic["limits_auto"] == "500000 1000000 100000"
    # a tile shape or order that is set acts from where it did before the column kernel
    assert logic["limits_tiles"] == "100000 100000"
    assert logic["limits_given"] == "0 7 7"
