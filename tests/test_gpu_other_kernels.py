"""The kernels that serve a call when the row kernels do not (no room for their
sample bits, a shape they leave alone), and the weld's 64-bit indices: the
tests that were written for them, with a context that is held to them."""
import pytest

from test_gpu_families import (reset_families, test_count_split_over_z,  # noqa: F401
                               test_family_long_z_segments, test_family_matches_oracle,
                               test_family_skips_empty_tiles)
from test_gpu_batch import (test_mixed_batch_matches_oracle,  # noqa: F401
                            test_repeated_batch_replays_graphs)
from test_gpu_large import (test_large_plane_in_a_batch,  # noqa: F401
                            test_planes_past_32bit_brick_offsets)
from test_gpu_weld import (test_weld_empty_and_small, test_weld_gpu_meshes,  # noqa: F401
                           test_weld_heavy_duplication, test_weld_large_table_skewed_x)
from test_gpu_weld_sizes import test_window_and_tile_ends  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def held(pkg):
    from importlib import import_module
    capi = import_module(pkg.__name__ + "._capi")
    ctx, limits = capi.context(0), (capi.MSH_LIMIT_SAMPLE_BITS, capi.MSH_LIMIT_WELD_INDEX32)

    def set_to(value):
        with ctx.lock:
            for what in limits:
                ctx.check(capi.lib().msh_set_limit(ctx.handle, what, value))

    set_to(0)
    yield
    set_to(-1)
