"""Units of the row kernels that several waves share (a surface that runs along
an x plane fills them): at the counts from which they are shared, where too
many are full, beside units that are not, alone and in batches, and in a
batch whose fields change between replays.  Against the oracle, exact."""
import numpy as np
import pytest

from helpers import assert_same_mesh, dev_field, noise

pytestmark = pytest.mark.gpu


def method_of(pkg, name):
    return {"mc": pkg.MarchingCubes, "mt": pkg.MarchingTetrahedra,
            "sn": pkg.NaiveSurfaceNets}[name](iso=0)


@pytest.fixture
def rows(pkg):
    # (some of these volumes go to the row kernels only when they are asked for)
    def reset(family):
        for name in ("mc", "mt", "sn"):
            for t in ("float32", "float64"):
                pkg.set_kernel_family(method_of(pkg, name), t, family)
    reset(2)
    yield
    reset(-1)


def plane(shape, dtype, at=0.31, bumps=0.0, seed=0):
    """A surface near x = at: whole planes of active cells, and some bumps."""
    x, y, z = (np.linspace(-1, 1, n) for n in shape)
    f = (x - at)[:, None, None] + np.zeros(shape)
    if bumps:
        f = f + bumps * np.sin((7 + seed) * y)[None, :, None] * np.cos(5 * z)[None, None, :]
    return f.astype(dtype)


def check(pkg, oracle, f, name):
    Vo, Fo = oracle.isosurface(f, name, iso=0)
    V, F = pkg.isosurface(dev_field(f), method_of(pkg, name))
    assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
    return len(Vo)


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nz", [4, 5, 7, 8, 9, 10, 13, 17, 25, 33, 34, 65])  # cells of a unit
def test_planes_at_the_counts(pkg, oracle, rows, name, dtype, nz):
    for ny in (65, 66, 100):
        for at in (0.31, -1.0, 1.0 - 1e-3):  # the first and the last x plane too
            assert check(pkg, oracle, plane((9, ny, nz), dtype, at, 0.004), name) > 0


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("nx", [34, 64, 80])  # 64: 8064 parts, 80: too many but by quarters
def test_many_full_units(pkg, oracle, rows, name, nx):
    f = np.random.default_rng(nx).standard_normal((nx, 129, 129)).astype(np.float32)
    assert check(pkg, oracle, f, name) > 100000


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
@pytest.mark.parametrize("nx", [2049, 2050, 4097, 4098, 8193, 8194])  # 2048, 4096, 8192 full units and one more
def test_most_shared_units(pkg, oracle, rows, name, nx):
    f = np.random.default_rng(nx).standard_normal((nx, 10, 33)).astype(np.float32)
    assert check(pkg, oracle, f, name) > 100000


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
def test_waves_of_several_units_skip_shared_ones(pkg, oracle, name):
    # a full unit between nearly empty ones, four units to a wave
    x = np.linspace(-1, 1, 513, dtype=np.float32)[:, None, None]
    yy = np.arange(16385) % 512
    s = np.where(yy // 64 == 1, 0, yy / 512 * 0.8 - 0.4).astype(np.float32)[None, :, None]
    f = np.empty((513, 16385, 17), np.float32, order="F")
    f[:] = x - np.float32(0.1) - s
    assert check(pkg, oracle, f, name) > 100000


@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
def test_batches(pkg, oracle, name):
    host = [plane((40, 70, 65), np.float32, 0.2, 0.01), noise((30, 40, 50), 1, np.float32),
            plane((20, 130, 33), np.float64, -0.4, 0.0), np.ones((9, 9, 9), np.float32),
            plane((33, 65, 129), np.float32, 0.7, 0.02, 3),
            np.random.default_rng(0).standard_normal((12, 66, 66)).astype(np.float32),
            np.random.default_rng(1).standard_normal((70, 129, 129)).astype(np.float64)]
    res = pkg.isosurface_batch([dev_field(f) for f in host], method_of(pkg, name))
    for f, (V, F) in zip(host, res):
        Vo, Fo = oracle.isosurface(f, name, iso=0)
        assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)


def test_replays_with_other_values(pkg, oracle):
    # the number of shared units changes from call to call at one set of buffers
    import torch
    shape, names = (24, 70, 70), ["mc", "mt", "sn"]
    sets = [[plane(shape, np.float32, 0.2 * i, 0.02 * j, i) for i in range(3)] for j in range(3)]
    sets.append([noise(shape, i, np.float32) for i in range(3)])
    sets.append([np.random.default_rng(i).standard_normal(shape).astype(np.float32) for i in range(3)])
    want = [[oracle.isosurface(f, n, iso=0) for f, n in zip(fs, names)] for fs in sets]
    fields = [dev_field(f) for f in sets[0]]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    for k in (0, 0, 0, 1, 1, 2, 3, 3, 3, 0, 4, 4, 4, 2, 0):
        for t, f in zip(fields, sets[k]):
            t.copy_(dev_field(f))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            res = pkg.isosurface_batch(fields, [method_of(pkg, n) for n in names])
        stream.synchronize()
        for (V, F), (Vo, Fo) in zip(res, want[k]):
            assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
