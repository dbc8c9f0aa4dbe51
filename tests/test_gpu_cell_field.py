"""GPU tests of the skip walk by cells (volumes larger than the caches) against
the stepping kernel that an explicitly requested raw layout runs, as the tests
of the walk by voxels do it: the same step counts, means within the rounding of
a few FP64 operations, over extents around multiples of a cell (4) and of a
field tile (32, 16, 16), labels at 2 bits and, with a bubble, at 4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make(shape, bubble, low_faces, seed):
    from anacor_public_amd import workload as W
    Z, Y, X = shape
    rng = np.random.default_rng(seed)
    z, y, x = (np.arange(n, dtype=np.float32) for n in shape)
    vol = np.zeros(shape, np.uint8)
    cyl = ((y[:, None] - Y / 2) / (0.48 * Y)) ** 2 + ((x[None] - X / 2) / (0.48 * X)) ** 2 <= 1
    vol[:, cyl] = 1
    vol[:, cyl & (np.abs(x[None] - X / 2) < X / 12)] = 2
    if bubble:
        vol[Z // 3:, cyl & (np.abs(y[:, None] - 0.7 * Y) < Y / 16)] = 4
    lo = [n // 3 for n in shape]
    hi = [2 * n // 3 for n in shape]
    vol[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] = 3
    coords = np.stack([rng.integers(a, b, 600) for a, b in zip(lo, hi)], 1)
    for corner in ((0, 0, 0), (Z - 1, Y - 1, X - 1)):
        vol[corner] = 3
    coords = np.concatenate([coords, [[Z - 1, Y - 1, X - 1]] + ([[0, 0, 0]] if low_faces else [])])
    s1, om = W.make_reflections(200, seed)
    wl = W.Workload("cells", vol, coords.astype(np.int64), s1, om)
    wl.voxel_size = np.array([0.3, 0.7, 1.1])
    wl.coefficients = np.array([0.011, 0.007, 0.019, 0.001])
    return wl


@pytest.mark.parametrize("shape", [(126, 782, 766), (127, 783, 767), (400, 417, 450),
                                   (1030, 254, 270), (17, 2046, 2040), (2045, 2046, 18)])
@pytest.mark.parametrize("bubble,low_faces", [(False, False), (True, False), (False, True)])
def test_equals_stepping(gpu, shape, bubble, low_faces):
    from anacor_public_amd import _lib
    from anacor_public_amd.ray_tracing import Tracer
    print(f"case: cells on {shape}, bubble={bubble}, low_faces={low_faces}", flush=True)
    assert np.prod(shape) > 64 << 20
    wl = make(shape, bubble, low_faces, sum(shape))
    with Tracer.for_workload(wl) as t:
        a32, sa = t.run_workload(wl), t.stats()["voxel_steps"]
        a64 = t.run_workload(wl, f64_mean=True)
        assert t.stats()["voxel_steps"] == sa
        ca = _lib.last_error()[0]
        t.set_layout(_lib.LAYOUT_RAW)
        b32, sb = t.run_workload(wl), t.stats()["voxel_steps"]
        b64 = t.run_workload(wl, f64_mean=True)
        assert ca == _lib.last_error()[0]
    assert sa == sb
    ok = ~np.isnan(b64)
    np.testing.assert_array_equal(np.isnan(a32), ~ok)
    np.testing.assert_array_equal(np.isnan(a64), ~ok)
    np.testing.assert_allclose(a64[ok], b64[ok], rtol=1e-13, atol=0)
    np.testing.assert_allclose(a32[ok], b32[ok], rtol=2.4e-7, atol=0)
