"""The order in which a single emit's blocks take the groups of shared units:
over 32 planes along x, then along the planes.  Planes of a number of units
that is no multiple of 8, last runs of fewer than 32 planes, planes with some
units shared and some not, and both lists.  Against the oracle, exact."""
import numpy as np
import pytest

from helpers import assert_same_mesh, dev_field

pytestmark = pytest.mark.gpu


@pytest.fixture
def rows(pkg):
    methods = (pkg.MarchingCubes, pkg.MarchingTetrahedra, pkg.NaiveSurfaceNets)
    for m in methods:
        pkg.set_kernel_family(m(iso=0), "float32", 2)
    yield
    for m in methods:
        pkg.set_kernel_family(m(iso=0), "float32", -1)


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("shape,dense", [
    ((34, 100, 170), 100),   # 10 units a plane, 33 planes of cells
    ((33, 100, 170), 100),   # 32
    ((70, 100, 170), 37),    # the rest of each plane is smooth
    ((130, 60, 100), 60),    # 4 units a plane
    ((66, 200, 200), 120),   # 22 units a plane
    ((210, 100, 200), 100),  # 11, too many parts but by quarters
])
def test_dense_planes(pkg, oracle, rows, name, shape, dense):
    f = np.random.default_rng(shape[0]).standard_normal(shape).astype(np.float32)
    f[:, dense:, :] = np.linspace(-1, 1, shape[0], dtype=np.float32)[:, None, None] - np.float32(0.123)
    Vo, Fo = oracle.isosurface(f, name, iso=0)
    method = {"mc": pkg.MarchingCubes, "mt": pkg.MarchingTetrahedra, "sn": pkg.NaiveSurfaceNets}[name](iso=0)
    V, F = pkg.isosurface(dev_field(f), method)
    assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
