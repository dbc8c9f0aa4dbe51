"""GPU test of calls that go up as one record (fewer than 8,192 reflections)
against a longer call, which goes up in parts: with one kernel (the raw layout's;
the automatic layout chooses by the call's size) and one tile size a
reflection's sums do not depend on the call it is in, so the means are the same
bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f64", [False, True])
def test_record_equals_parts(gpu, f64):
    from anacor_public_amd import _lib
    from anacor_public_amd import workload as W
    from anacor_public_amd.ray_tracing import Tracer
    wl = W.small_config(R=8193)
    with Tracer.for_workload(wl) as t:
        t.set_layout(_lib.LAYOUT_RAW)
        t.set_tile(512)
        whole = t.run_workload(wl, f64_mean=f64)
        steps = t.stats()["voxel_steps"]
        for n in (8191, 1, 8192, 257, 256):
            print(f"case: {n} reflections, f64={f64}", flush=True)
            part = t.run_workload(wl.subset(n), f64_mean=f64)
            np.testing.assert_array_equal(part.view(np.uint64), whole[:n].view(np.uint64))
            assert 0 < t.stats()["voxel_steps"] < steps
