"""Volumes of many short x planes, at the sizes from which they go to the row
kernels: alone and in a batch beside volumes that do.  Against the oracle,
exact."""
import numpy as np
import pytest

from helpers import assert_same_mesh, dev_field, noise

pytestmark = pytest.mark.gpu

SHAPES = [(1024, 3, 9), (1025, 2, 16), (1025, 2, 17), (1025, 3, 9),  # 1024 units; 15 and 16 cells
          (4096, 2, 3), (4097, 2, 3), (4096, 4, 20), (4097, 4, 20),  # 4096 units
          (4097, 13, 6), (4097, 12, 6), (4097, 9, 9), (4097, 10, 17), (4097, 10, 18),  # 60 cells, 10 rows, 16 long
          (4097, 17, 33), (4097, 17, 32), (4097, 33, 33), (4097, 33, 32),  # 512 and 1024 cells
          (4500, 70, 2)]  # two units a plane


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("shape", SHAPES)
def test_sizes(pkg, oracle, shape, name):
    m = {"mc": pkg.MarchingCubes, "mt": pkg.MarchingTetrahedra, "sn": pkg.NaiveSurfaceNets}[name](iso=0)
    f = noise(shape, sum(shape), np.float32)
    Vo, Fo = oracle.isosurface(f, name, iso=0)
    V, F = pkg.isosurface(dev_field(f), m)
    assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)


def test_batch(pkg, oracle):
    names = ["mc", "mt", "sn"]
    host = [noise(s, i, np.float64 if i % 4 == 0 else np.float32)
            for i, s in enumerate(SHAPES + [(30, 31, 32), (2, 2, 2), (20, 40, 50)])]
    make = {"mc": pkg.MarchingCubes, "mt": pkg.MarchingTetrahedra, "sn": pkg.NaiveSurfaceNets}
    res = pkg.isosurface_batch([dev_field(f) for f in host],
                               [make[names[i % 3]](iso=0) for i in range(len(host))])
    for i, (f, (V, F)) in enumerate(zip(host, res)):
        Vo, Fo = oracle.isosurface(f, names[i % 3], iso=0)
        assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
