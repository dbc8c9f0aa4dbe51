"""GPU tests of reflections that the skip walk leaves to the stepping kernel: at
rotation angles of 270 degrees the beam lies within 1e-16 of an axis, where a
stepped coordinate is too close to a boundary for the walk's table.  Calls of
such reflections only, of some, and of none, through every way a call is sent
(one record, two parts, without allocation, a batch, a batch as a graph): the
same bits, step counts and numbers of retraced reflections as each other, and
means within the rounding of a few FP64 operations of the stepping kernel's."""
import ctypes as ct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (60, 90, 110)           # extents that take the walk whatever the call's size


def make(R, marked, seed):
    """marked: the share of reflections at 270 degrees."""
    from anacor_public_amd import workload as W
    rng = np.random.default_rng(seed)
    g = np.indices(SHAPE)
    vol = (np.hypot(g[1] - 45, g[2] - 55) <= 44).astype(np.uint8)
    vol[(vol == 1) & (np.abs(g[2] - 55) < 4)] = 2
    vol[20:40, 30:60, 40:75] = 3
    co = np.argwhere(vol == 3)
    s1, om = W.make_reflections(R, seed)
    om[rng.random(R) < marked] = 1.5 * np.pi
    wl = W.Workload("retraced", vol, co[rng.permutation(len(co))[:300]], s1, om)
    wl.voxel_size = np.array([0.3, 0.7, 1.1])
    wl.coefficients = np.array([0.011, 0.007, 0.019, 0.001])
    return wl


def bits(a):
    return np.ascontiguousarray(a, np.float64).view(np.uint64)


@pytest.mark.parametrize("marked", [0.0, 0.1, 1.0])
@pytest.mark.parametrize("R", [1, 255, 257, 3000, 8192, 9001])
@pytest.mark.parametrize("f64", [False, True])
def test_every_way(gpu, R, marked, f64):
    from anacor_public_amd import _lib
    from anacor_public_amd.ray_tracing import Batch, Tracer
    print(f"case: {R} reflections, {marked} at 270 degrees, f64={f64}", flush=True)
    wl = make(R, marked, R + 7)
    n = int(np.count_nonzero(wl.omega == 1.5 * np.pi))
    with Tracer.for_workload(wl) as t:
        t.set_tile(256)
        a, sa = t.run_workload(wl, f64_mean=f64), t.stats()["voxel_steps"]
        assert t.last_walk() == (_lib.WALK_VOXELS, n)
        again = t.run_workload(wl, f64_mean=f64)
        assert t.stats()["voxel_steps"] == sa
        np.testing.assert_array_equal(bits(again), bits(a))
        p = lambda v: np.ascontiguousarray(v, np.float64).ctypes.data_as(ct.c_void_p)  # noqa: E731
        na = np.empty(R)
        keep = [np.ascontiguousarray(v, np.float64) for v in (wl.s1, wl.omega, wl.raw_xray,
                                                               wl.omega_axis, wl.F)]
        assert gpu.anacor_ctx_run_noalloc(t.handle, p(keep[0]), p(keep[1]), R, p(keep[2]),
                                          p(keep[3]), p(keep[4]),
                                          _lib.FLAG_F64_MEAN if f64 else 0, p(na)) == 0
        assert t.stats()["voxel_steps"] == sa and t.last_walk() == (_lib.WALK_VOXELS, n)
        np.testing.assert_array_equal(bits(na), bits(a))
        t.set_layout(_lib.LAYOUT_RAW)
        b, sb = t.run_workload(wl, f64_mean=f64), t.stats()["voxel_steps"]
        assert t.last_walk() == (_lib.WALK_STEPS, 0)
    assert sa == sb
    np.testing.assert_allclose(a, b, rtol=1e-13 if f64 else 2.4e-7, atol=0)
    with Batch([wl, wl]) as bt:
        for i in range(2):
            bt.sample(i).set_tile(256)
        for graph in (False, True):
            bt.set_graph(graph)
            for _ in range(2):
                outs = bt.run([wl.s1] * 2, [wl.omega] * 2, wl.raw_xray, wl.omega_axis, wl.F,
                              f64_mean=f64)
                assert bt.stats()["voxel_steps"] == 2 * sa
                for i, o in enumerate(outs):
                    np.testing.assert_array_equal(bits(o), bits(a))
                    assert bt.sample(i).last_walk() == (_lib.WALK_VOXELS, n)
