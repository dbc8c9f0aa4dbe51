"""GPU tests of the skip walk on crystals cut by the volume's low faces (a cropped
volume): the reference ends a ray that starts on a low face at once, also where
it leads away from it, or aborts there.  The walk covers these rays itself, so
no reflection of random directions is left to the stepping kernel; the same
errors and step counts, and means within the rounding of a few FP64 operations,
as in the walk's other tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make(shape, low):
    """A crystal ball around the corner, edge or face at coordinate 0 of the axes in
    `low`, in a liquor cylinder with a loop."""
    from anacor_public_amd import workload as W
    rng = np.random.default_rng(sum(shape) + len(low))
    c = [0 if i in low else n // 2 for i, n in enumerate(shape)]
    g = np.indices(shape)
    vol = np.ones(shape, np.uint8)
    vol[:, np.hypot(g[1][0] - shape[1] / 2, g[2][0] - shape[2] / 2) > 0.6 * max(shape[1:])] = 0
    vol[(vol == 1) & (np.abs(g[2] - shape[2] // 2) < 3)] = 2
    vol[sum(((a - b) / (0.3 * n)) ** 2 for a, b, n in zip(g, c, shape)) <= 1] = 3
    co = np.argwhere(vol == 3)
    co = co[rng.permutation(len(co))[:900]]
    face = np.argwhere((vol == 3) & np.logical_or.reduce([g[a] == 0 for a in low]))
    co = np.concatenate([co, face[:100]]).astype(np.int64)
    s1, om = W.make_reflections(1200, sum(shape))
    wl = W.Workload("low", vol, co, s1, om)
    wl.voxel_size = np.array([0.3, 0.7, 1.1])
    wl.coefficients = np.array([0.011, 0.007, 0.019, 0.001])
    return wl


@pytest.mark.parametrize("low", [(0,), (1,), (2,), (0, 1), (1, 2), (0, 1, 2)])
@pytest.mark.parametrize("shape", [(48, 50, 52), (65, 64, 33)])
def test_trace(gpu, shape, low):
    from anacor_public_amd import _lib
    from anacor_public_amd.ray_tracing import Tracer
    print(f"case: crystal at the low faces {low} of {shape}", flush=True)
    wl = make(shape, low)
    with Tracer.for_workload(wl) as t:
        a, sa = t.run_workload(wl, f64_mean=True), t.stats()["voxel_steps"]
        walk, retraced = t.last_walk()
        ea = _lib.last_error()
        t.set_layout(_lib.LAYOUT_RAW)
        b, sb = t.run_workload(wl, f64_mean=True), t.stats()["voxel_steps"]
        eb = _lib.last_error()
    assert ea == eb
    assert walk == _lib.WALK_VOXELS
    assert sa == sb
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    ok = ~np.isnan(b)
    assert ok.any() or len(low) > 1     # on two low faces the reference aborts nearly always
    np.testing.assert_allclose(a[ok], b[ok], rtol=1e-13, atol=0)
    assert retraced == 0


def test_map(gpu):
    from anacor_public_amd import _lib
    from anacor_public_amd.gridding import Gridding
    from anacor_public_amd.ray_tracing import Tracer
    print("case: map of a crystal at all low faces", flush=True)
    wl = make((48, 50, 52), (0, 1, 2))
    maps = []
    for layout in (_lib.LAYOUT_AUTO, _lib.LAYOUT_RAW):
        with Tracer.for_workload(wl) as t:
            t.set_layout(layout)
            with Gridding(t, 71, 37) as g:
                maps.append(g.map())
                if layout == _lib.LAYOUT_AUTO:
                    walk, retraced = t.last_walk()
    assert walk == _lib.WALK_VOXELS
    np.testing.assert_allclose(maps[0], maps[1], rtol=1.2e-7, atol=0, equal_nan=True)
    # left over: the directions on the planes where the tracer's rules switch
    assert retraced < 0.25 * len(maps[0])
