"""GPU test of the skip walk on directions with components of exactly zero.  The
angles of such a direction can be those of one slightly off (a zero x component
counts as 0.001), so its rays drift along that axis, towards either side, while
the direction itself has no side there.  Voxels on every surface of a crystal
block, against the stepping kernel that an explicitly requested raw layout
runs: the same step counts, means within the rounding of a few FP64
operations, as in the walk's other tests."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COMPONENTS = [v for v in itertools.product((0.0, 0.6, -0.6, 1.0, -1.0), repeat=3)
              if 0.0 in v and any(v)]


@pytest.mark.parametrize("shape", [(40, 44, 48), (60, 248, 30), (31, 33, 300)])
def test_equals_stepping(gpu, shape):
    from anacor_public_amd import _lib
    from anacor_public_amd import workload as W
    from anacor_public_amd.ray_tracing import Tracer
    print(f"case: directions with zero components on {shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    lo = np.array(shape) // 3
    hi = 2 * np.array(shape) // 3
    vol = np.ones(shape, np.uint8)
    vol[tuple(slice(a, b) for a, b in zip(lo, hi))] = 3
    coords = []
    for axis in range(3):                      # surfaces of the block
        for side in (lo[axis], hi[axis] - 1):
            c = np.stack([rng.integers(a, b, 300) for a, b in zip(lo, hi)], 1)
            c[:, axis] = side
            coords.append(c)
    coords = np.concatenate(coords).astype(np.int64)
    s1 = np.array(COMPONENTS)
    s1 = np.tile(s1, (-(-(1 << 20) // (len(coords) * len(s1))) + 1, 1))
    assert len(s1) * len(coords) > 1 << 20     # the walk's calls, whatever the extents
    wl = W.Workload("zero", vol, coords, np.ascontiguousarray(s1), np.zeros(len(s1)))
    wl.voxel_size = np.array([0.3, 0.7, 1.1])
    wl.coefficients = np.array([0.011, 0.007, 0.019, 0.001])
    with Tracer.for_workload(wl) as t:
        a, sa = t.run_workload(wl, f64_mean=True), t.stats()["voxel_steps"]
        t.set_layout(_lib.LAYOUT_RAW)
        b, sb = t.run_workload(wl, f64_mean=True), t.stats()["voxel_steps"]
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    ok = ~np.isnan(b)
    assert ok.any()
    np.testing.assert_allclose(a[ok], b[ok], rtol=1e-13, atol=0)
    assert sa == sb
