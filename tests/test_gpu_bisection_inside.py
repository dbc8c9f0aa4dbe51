"""GPU test of the bisection's search for rays that stay inside the volume
(extents of at most 1,024) against the FP64 oracle, bit for bit per ray: extents
at and around the limit, thin volumes whose rays leave after a step or none,
and num_cls 4 with a bubble."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1024, 9, 12), (1025, 9, 12), (3, 40, 1023), (2, 2, 2),
                                   (33, 64, 95)])
@pytest.mark.parametrize("num_cls", [3, 4])
def test_lengths_match_oracle(gpu, oracle, shape, num_cls):
    from anacor_public_amd import workload as W
    from anacor_public_amd.ray_tracing import Tracer
    print(f"case: bisection on {shape}, num_cls {num_cls}", flush=True)
    rng = np.random.default_rng(sum(shape))
    Z, Y, X = shape
    z, y, x = np.indices(shape)
    vol = np.ones(shape, np.uint8)
    vol[np.abs(x - X // 2) < max(1, X // 6)] = 2
    vol[y < Y // 8] = 0
    if num_cls == 4:
        vol[np.abs(z - 3 * Z // 4) < max(1, Z // 10)] = 4
    vol[Z // 4:Z // 2 + 1, Y // 4:Y // 2 + 1, X // 4:X // 2 + 1] = 3
    coords = np.argwhere(vol == 3)
    coords = coords[rng.permutation(len(coords))[:60]]
    wl = W.Workload("inside", vol, coords, *W.make_reflections(24, 11))
    rs, xr = rng.normal(size=(24, 3)), rng.normal(size=(24, 3))
    rs /= np.linalg.norm(rs, axis=1, keepdims=True)
    xr /= np.linalg.norm(xr, axis=1, keepdims=True)
    with Tracer.for_workload(wl) as t:
        A, L = t.bisection_rotated(rs, xr, num_cls=num_cls, f64_mean=True, lengths=True)
    for i in range(24):
        mean, _, Lo = oracle.ib_test(wl, wl.coords, rs[i], xr[i], num_cls, lengths=True)
        if np.isnan(mean):
            assert np.isnan(A[i])
            continue
        np.testing.assert_array_equal(L[i], Lo)
        np.testing.assert_allclose(A[i], mean, rtol=1e-12, atol=0)
