"""Which kernels a call takes: from the row kernels to the others and back because
of the room for the sample bits, at the same buffers, and because of the axes;
the meshes stay those of the oracle.  Exact."""
import numpy as np
import pytest

from helpers import assert_same_mesh, dev_field, noise

pytestmark = pytest.mark.gpu


@pytest.fixture
def set_limit(pkg):
    from importlib import import_module
    capi = import_module(pkg.__name__ + "._capi")
    ctx = capi.context(0)

    def set_to(what, value):
        with ctx.lock:
            ctx.check(capi.lib().msh_set_limit(ctx.handle, what, value))

    yield set_to
    set_to(capi.MSH_LIMIT_SAMPLE_BITS, -1)


def test_unknown_limit_is_refused(set_limit):
    with pytest.raises(ValueError):
        set_limit(9, 0)


def test_repeated_batch_changes_kernels(pkg, oracle, set_limit):
    # the same batch by the row kernels, then with no room for their bits,
    # then with room again, each often enough to be captured and replayed;
    # the workspaces keep their addresses (they only grow)
    import torch
    shapes = [(33, 34, 35), (20, 50, 70), (64, 9, 40), (2, 3, 130)]
    names = ["mc", "mt", "sn", "mc"]
    methods = [pkg.MarchingCubes(iso=0), pkg.MarchingTetrahedra(iso=0), pkg.NaiveSurfaceNets(iso=0),
               pkg.MarchingCubes(iso=0)]
    host = [noise(s, i, np.float32 if i % 2 else np.float64) for i, s in enumerate(shapes)]
    want = [oracle.isosurface(f, n, iso=0) for f, n in zip(host, names)]
    fields = [dev_field(f) for f in host]
    stream = torch.cuda.Stream()  # (the null stream is never captured)
    torch.cuda.synchronize()
    for limit in (-1, 0, -1, 0):
        set_limit(0, limit)
        for rep in range(4):
            with torch.cuda.stream(stream):
                res = pkg.isosurface_batch(fields, methods)
            stream.synchronize()
            for (V, F), (Vo, Fo) in zip(res, want):
                assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
            del res
            torch.cuda.synchronize()


@pytest.mark.parametrize("limit", [-1, 0])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name", ["mc", "mt", "sn"])
def test_axes_without_finite_ends(pkg, oracle, set_limit, name, dtype, limit):
    # p + mu * (p - p) is NaN for an infinite p, whatever mu is
    set_limit(0, limit)
    m = {"mc": pkg.MarchingCubes(iso=0), "mt": pkg.MarchingTetrahedra(iso=0),
         "sn": pkg.NaiveSurfaceNets(iso=0)}[name]
    f = noise((9, 10, 40), 5, dtype)
    inf, one, big = np.inf, (-1, 1), np.finfo(np.float64).max
    for ax in (((-1.0, inf), one, one), (one, (-inf, 1.0), (np.float32(-1), np.float32(inf))),
               (one, one, (np.nan, 1.0)), ((-big, big), one, (-inf, inf)),
               ((np.float32(-3e38), np.float32(3e38)), one, one)):
        Vo, Fo = oracle.isosurface(f, name, iso=0, X=ax[0], Y=ax[1], Z=ax[2])
        V, F = pkg.isosurface(dev_field(f), m, *ax)
        assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
        (V, F), = pkg.isosurface_batch([dev_field(f)], m, [ax])
        assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)


def test_families_mix_in_a_batch(pkg, oracle):
    # each volume of a batch runs its own class's family: the row kernels for
    # some, every other family beside them, and a volume nothing crosses
    import torch
    make = {"mc": pkg.MarchingCubes, "mt": pkg.MarchingTetrahedra, "sn": pkg.NaiveSurfaceNets}
    types = [(n, t) for n in make for t in ("float32", "float64")]
    host = [noise((20 + 3 * i, 33 + i, 30 + 7 * i), i, t) for i, (n, t) in enumerate(types * 2)]
    host.append(np.ones((9, 8, 70), np.float32))
    names = [n for n, _ in types * 2] + ["mt"]
    fields, methods = [dev_field(f) for f in host], [make[n](iso=0) for n in names]
    want = [oracle.isosurface(f, n, iso=0) for f, n in zip(host, names)]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        for shift in range(4):
            for i, (n, t) in enumerate(types):
                pkg.set_kernel_family(make[n](iso=0), t, [-1, 0, 2, 1, -1, 3][(i + shift) % 6])
            for rep in range(3):
                with torch.cuda.stream(stream):
                    res = pkg.isosurface_batch(fields, methods)
                stream.synchronize()
                for (V, F), (Vo, Fo) in zip(res, want):
                    assert_same_mesh(V.cpu().numpy(), F.cpu().numpy(), Vo, Fo)
    finally:
        for n, t in types:
            pkg.set_kernel_family(make[n](iso=0), t, -1)
