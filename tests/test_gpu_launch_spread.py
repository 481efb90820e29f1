"""The megakernel's split of a launch's paths over its wavefronts: launches
with fewer paths than wavefronts, one path per wavefront, a few lanes per
wavefront, exactly one path per lane and more (paths beyond the first ones are
claimed through counters), at sizes with partial tiles, against the oracle bit
for bit."""
import numpy as np
import pytest

import vpo
from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu

# (workgroup, workgroups per CU): 256 wavefronts, and the default shape
SHAPES = {"small": (64, 1), "default": (0, 0)}
# width, height, spp (camera paths are padded to 8x8 tiles): 64 paths; 192;
# 4096 (one per wavefront of the default shape); 16384 (one per lane of the
# small shape); 20480 and 65280 (claimed beyond that); 1 pixel deep in samples
SIZES = [(1, 1, 1), (9, 7, 3), (64, 64, 1), (64, 32, 8), (40, 32, 16), (40, 23, 68), (1, 1, 300)]


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("size", SIZES)
def test_paths_spread_over_wavefronts(ctx, size, shape):
    w, h, spp = size
    rows = scenes.random_scene(40, 5, albedo=0.9)
    env = scenes.sky_env(64, 32, sun_radius_deg=4.0, sun_scale=50.0)
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    p = volprim.default_params(width=w, height=h, spp=spp, seed=3, max_depth=24, phase_g=0.3, use_ris=spp % 2)
    print(f"[case] launch spread {w}x{h}x{spp}, {shape} shape", flush=True)
    sc, ev = ctx.scene(rows), ctx.env(env)
    _, _, rec, _ = sc.export()
    block, per_cu = SHAPES[shape]
    launch = volprim.LaunchConfig(block, per_cu, 0, 0, 0, volprim.PIPELINE_MEGAKERNEL, 0)
    img = ctx.render_jobs([(sc, ev, cam, p)], launch=launch)[0][0]
    sc.close()
    ev.close()
    ref, _, _ = vpo.render(rec, env, cam.pod(), w, h, spp, seed=3, max_depth=24, phase_g=0.3, use_ris=bool(spp % 2))
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
