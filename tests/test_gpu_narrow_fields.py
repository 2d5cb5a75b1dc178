"""Sample bits of fields of up to 32 columns along x, at the ends of their tiles
(256 columns by 4 words) and where they begin, alone and in a batch.  Against
the oracle, exact."""
import numpy as np
import pytest

from helpers import assert_same_mesh, dev_field, noise

pytestmark = pytest.mark.gpu

SHAPES = [(32, 256, 1000), (33, 256, 1000), (32, 255, 1000), (31, 1100, 180), (2, 8191, 127), (3, 5500, 130),
          (2, 32769, 129), (5, 13108, 33), (17, 3856, 31), (16, 4095, 100)]


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES)
def test_sizes(pkg, oracle, shape, dtype, name):
    m = {"mc": pkg.MarchingCubes, "mt": pkg.MarchingTetrahedra, "sn": pkg.NaiveSurfaceNets}[name](iso=0)
    pkg.set_kernel_family(m, dtype, 2)
    f = (noise(shape, sum(shape), np.float32) - np.float32(0.6)).astype(dtype)
    f[1, ::97, ::41] = np.nan
    Vo, Fo = oracle.isosurface(f, name, iso=0)
    assert len(Fo) > 100
    try:
        V, F = pkg.isosurface(dev_field(f), m)
        assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
        (V, F), (V2, F2) = pkg.isosurface_batch([dev_field(f), dev_field(f[:, :40, :50].copy())], m)
        assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
    finally:
        pkg.set_kernel_family(m, dtype, -1)
