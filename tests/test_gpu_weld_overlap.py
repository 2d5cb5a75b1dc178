"""msh_weld_to refuses a face output that partly overlaps the faces (threads
would read indices that others have renumbered) before anything runs."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [8, 24, 48 - 8, -8, -40])
def test_partial_overlap_is_refused(pkg, shift):
    import torch
    from importlib import import_module
    capi = import_module(pkg.__name__ + "._capi")
    V = torch.zeros((4, 3), dtype=torch.float64, device="cuda")
    out = torch.empty_like(V)
    buf = torch.ones(64, dtype=torch.int64, device="cuda")
    F = buf.data_ptr() + 8 * 24  # two faces, 48 bytes
    ctx, n = capi.context(0), ctypes.c_int64()
    args = lambda o: (ctx.handle, capi.MSH_FLOAT64, 4, ctypes.c_void_p(V.data_ptr()), 2,  # noqa: E731
                      ctypes.c_void_p(F), ctypes.c_void_p(o), ctypes.c_void_p(out.data_ptr()),
                      ctypes.byref(n))
    with ctx.lock:
        assert capi.lib().msh_weld_to(*args(F + shift)) == capi.MSH_ERR_ARGUMENT
        for apart in (F, F + 48, F - 48):  # itself, and right behind and before
            assert capi.lib().msh_weld_to(*args(apart)) == capi.MSH_OK
            assert n.value == 1
