"""The row kernels (sample bits, counts and emits that go by words of 32 samples
along z and units of 64 words) at the sizes where their tilings end: against
the oracle, faces identical and vertices bit-identical.  No tolerance."""
import numpy as np
import pytest

from helpers import assert_same_mesh, dev_field, noise

pytestmark = pytest.mark.gpu


def method_of(pkg, name, iso=0):
    return {"mc": pkg.MarchingCubes, "mt": pkg.MarchingTetrahedra,
            "sn": pkg.NaiveSurfaceNets}[name](iso=iso)


def check(pkg, oracle, f, name, iso=0, axes=((-1, 1),) * 3):
    Vo, Fo = oracle.isosurface(f, name, iso=iso, X=axes[0], Y=axes[1], Z=axes[2])
    # (small tetrahedra volumes go to the row kernels only when these are asked for)
    for family in (2, -1) if name == "mt" else (-1,):
        pkg.set_kernel_family(method_of(pkg, name), str(f.dtype), family)
        V, F = pkg.isosurface(dev_field(f), method_of(pkg, name, iso), *axes)
        assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
    return len(Fo)


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [
    (2, 2, 2), (3, 2, 33), (2, 3, 32), (5, 4, 31),  # one word of cells a row; 33: two of samples
    (6, 7, 34), (4, 9, 65), (5, 6, 66), (7, 5, 97),  # word ends along z
    (64, 3, 40), (65, 4, 5), (128, 3, 33), (129, 2, 40), (131, 5, 36),  # tile ends along x
    (9, 65, 30), (5, 64, 31), (6, 66, 20), (4, 23, 97), (3, 130, 70),  # unit ends along (y, z)
    (3, 4, 3850), (2, 3, 4200),  # rows of 121 and 132 words: longer than the short-row division
])
def test_tiling_ends(pkg, oracle, shape, dtype, name):
    check(pkg, oracle, noise(shape, sum(shape), dtype), name)


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_every_cell_active(pkg, oracle, dtype, name):
    # white noise: units of up to 2048 active cells, the queue fills many times
    f = np.random.default_rng(3).standard_normal((19, 37, 100)).astype(dtype)
    assert check(pkg, oracle, f, name, 0.1) > 100000


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
def test_level_types_and_axes(pkg, oracle, name):
    f = noise((33, 35, 67), 4, np.float32)
    axes = (((np.float32(-1.5), np.float32(2.25)),) * 3, ((0, 10), (np.float32(-0.3), np.float32(0.7)), (-2.5, 3.0)))
    for iso in (0, np.float32(0.05), -0.05):
        for ax in axes:
            check(pkg, oracle, f, name, iso, ax)


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
def test_values_without_order(pkg, oracle, name):
    # NaN, infinities and equal neighbours at the level
    rng = np.random.default_rng(8)
    f = noise((20, 21, 70), 5, np.float32)
    for v in (np.nan, np.inf, -np.inf, 0.0, -0.0):
        f[tuple(rng.integers(0, n, 40) for n in f.shape)] = v
    check(pkg, oracle, f, name)


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
def test_sparse_units(pkg, oracle, name):
    # 129 units an x plane and few vertices a unit: waves that take several
    # units, with a remainder, most of them empty
    x = np.linspace(-1, 1, 2049)[:, None, None]
    y = np.linspace(-1, 1, 8200)[None, :, None]
    z = np.linspace(0, 1, 2)[None, None, :]
    f = np.asfortranarray((np.sqrt(x * x + y * y) - 0.5 + 0.001 * z).astype(np.float32))
    assert check(pkg, oracle, f, name) > 1000


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("nx", [2049, 2050])  # 2048 units, scanned by the count's last block, and one more
def test_scan_in_the_count(pkg, oracle, nx, name):
    for seed in (1, 2):
        assert check(pkg, oracle, noise((nx, 65, 5), seed, np.float32), name) > 1000


@pytest.mark.parametrize("dtype,shape", [
    (np.float32, (200, 20000, 36)), (np.float64, (250, 800, 347)),  # tiles of 256 columns
    (np.float32, (301, 910, 500)), (np.float64, (40, 53000, 33)),  # tiles of 128
])
def test_field_beyond_the_cache(pkg, oracle, dtype, shape):
    # over 512 MiB, with ends of tiles along x and of words along z
    x, y, z = (np.linspace(-1, 1, n, dtype=dtype) for n in shape)
    f = np.empty(shape, dtype, order="F")
    f[:] = np.sin(400 * y)[None, :, None] * x[:, None, None] + dtype(0.3) * z - dtype(0.9)
    assert check(pkg, oracle, f, "mc") > 1000
