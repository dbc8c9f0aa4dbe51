"""GPU tests of what a context holds when the skip walk's field is not for it: a
listed voxel of another label than 3, or tables larger than a workgroup's LDS.
Such a context takes no more device memory than one that never asks for a field
(full_iteration), and its traces step.  Volumes past 160 MB, whose field has
parts of its own beside the octants."""
import ctypes as ct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = ct.CDLL("libamdhip64.so")
    free, total = ct.c_size_t(), ct.c_size_t()
    assert hip.hipMemGetInfo(ct.byref(free), ct.byref(total)) == 0
    return free.value


def workload(shape, other_label, full):
    from anacor_public_amd import workload as W
    rng = np.random.default_rng(sum(shape))
    vol = np.full(shape, 3, np.uint8)
    # voxels at both ends of every axis, so that the tables span the volume
    ends = np.array([[0, 0, 0], [n - 1 for n in shape]])
    co = np.concatenate([ends, np.stack([rng.integers(1, n - 1, 500) for n in shape], 1)])
    if other_label:
        vol[tuple(co[-1])] = 1
    s1, om = W.make_reflections(16, 3)
    wl = W.Workload("memory", vol, co.astype(np.int64), s1, om)
    wl.full_iteration = full
    return wl


@pytest.mark.parametrize("shape,other_label", [((551, 552, 553), True), ((2046, 2046, 76), False)])
def test_no_field_no_memory(gpu, shape, other_label):
    from anacor_public_amd import _lib
    from anacor_public_amd.ray_tracing import Tracer
    print(f"case: context without a field on {shape}", flush=True)
    with Tracer.for_workload(workload((8, 8, 8), False, 1)):
        used = []
        for full in (1, 0):
            wl = workload(shape, other_label, full)
            before = free_bytes()
            with Tracer.for_workload(wl) as t:
                used.append(before - free_bytes())
                if not full:
                    t.run_workload(wl)
                    assert t.last_walk() == (_lib.WALK_STEPS, 0)
        assert used[1] <= used[0] + (4 << 20)   # the allocator's granularity, twice
