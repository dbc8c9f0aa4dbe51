"""bench.py's roofline record, on the CPU: a rate of bytes and its share of the
memory's peak for the stepping kernel only, whose every voxel step reads a byte;
the walk by free distances reads one byte for many steps and reports none."""
import os
import sys

import pytest

from conftest import ROOT

sys.path.insert(0, ROOT)

import bench  # noqa: E402

from anacor_public_amd import _lib  # noqa: E402

STEPS = 101_723_984_094


@pytest.mark.parametrize("walks,kernel", [
    ({_lib.WALK_VOXELS}, "skip_kernel"), ({_lib.WALK_CELLS}, "skip_kernel"),
    ({_lib.WALK_VOXELS, _lib.WALK_STEPS}, "skip_kernel and trace_kernel")])
def test_no_rate_of_bytes_for_the_walk(walks, kernel):
    r = bench.trace_roofline(walks, 14.0, STEPS, 0.02 * STEPS, False)
    assert r["kernel"] == kernel and r["kernel_ms"] == 14.0
    assert [r[k] for k in ("achieved", "frac", "traffic", "bytes_per_launch")] == [None] * 4
    assert r["voxel_steps_per_launch"] == STEPS


def test_stepping_kernel():
    r = bench.trace_roofline({_lib.WALK_STEPS}, 62.5, STEPS, 5.0, True)
    assert r["kernel"] == "trace_kernel, one launch per sample"
    assert r["achieved"] == pytest.approx(STEPS / 62.5e-3 / 1e9)
    assert r["frac"] == pytest.approx(r["achieved"] / 8000.0)
    assert r["bytes_per_launch"] == STEPS and r["traffic"] == 5.0
