"""GPU tests of the absorption map by the skip walk (the automatic layout)
against the stepping kernel (an explicitly requested raw layout): the same FP32
values but for a rounding of FP64 sums that differ in their last bits (one unit
in the last place), the same NaN entries, with directions on the planes where
the tracer's rules switch (theta and phi at multiples of 45 degrees), which the
skip walk leaves to the stepping kernel."""
import numpy as np
import pytest

from test_gpu_skip_walk import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,grid", [((33, 47, 61), (72, 48)), ((64, 64, 64), (72, 48)),
                                        ((100, 66, 130), (120, 60)), ((95, 33, 97), (71, 37))])
@pytest.mark.parametrize("low_faces", [False, True])
def test_map_equals_stepping(gpu, shape, grid, low_faces):
    from anacor_public_amd import _lib
    from anacor_public_amd.gridding import Gridding
    from anacor_public_amd.ray_tracing import Tracer
    print(f"case: map on {shape}, grid {grid}, low_faces={low_faces}", flush=True)
    wl = make(shape, 3, low_faces=low_faces)
    maps = []
    for layout in (_lib.LAYOUT_AUTO, _lib.LAYOUT_RAW):
        with Tracer.for_workload(wl) as t:
            t.set_layout(layout)
            with Gridding(t, *grid) as g:
                maps.append(g.map())
    np.testing.assert_allclose(maps[0], maps[1], rtol=1.2e-7, atol=0, equal_nan=True)
