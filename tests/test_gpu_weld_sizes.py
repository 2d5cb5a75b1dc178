"""Vertex welding at the ends of its windows (1024 vertices), prefix tiles (4096)
and table sizes, through both entry points (faces renumbered in place, and
into another buffer), against the definition: exact."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nv", [1, 2, 511, 512, 513, 1023, 1024, 1025, 4095, 4096, 4097, 13107, 70001])
def test_window_and_tile_ends(pkg, oracle, nv, dtype):
    import torch
    from importlib import import_module
    capi = import_module(pkg.__name__ + "._capi")
    rng = np.random.default_rng(nv)
    # about a third of the vertices are copies, near and far
    V = rng.integers(0, max(2, nv // 3), (nv, 1)).astype(dtype) + np.array([[0, 0.5, -0.0]], dtype)
    F = rng.integers(1, nv + 1, (2 * nv + 1, 3)).astype(np.int64)
    Vo, Fo = oracle.weld(V, F)
    v, f = torch.from_numpy(V).cuda(), torch.from_numpy(F).cuda()
    Vw, Fw = pkg.weld(v, f)
    assert torch.equal(f.cpu(), torch.from_numpy(F))  # the arguments stay as they are
    assert np.array_equal(Vw.cpu().numpy().view(np.uint8), Vo.view(np.uint8))
    assert np.array_equal(Fw.cpu().numpy(), Fo)
    # in place
    L, ctx = capi.lib(), capi.context(0)
    out, n = torch.empty_like(v), ctypes.c_int64()
    with ctx.lock:
        ctx.check(L.msh_set_stream(ctx.handle, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        ctx.check(L.msh_weld(ctx.handle, capi.MSH_FLOAT32 if dtype == np.float32 else capi.MSH_FLOAT64,
                             nv, ctypes.c_void_p(v.data_ptr()), len(F), ctypes.c_void_p(f.data_ptr()),
                             ctypes.c_void_p(out.data_ptr()), ctypes.byref(n)))
    assert n.value == len(Vo)
    assert np.array_equal(out[:n.value].cpu().numpy().view(np.uint8), Vo.view(np.uint8))
    assert np.array_equal(f.cpu().numpy(), Fo)
