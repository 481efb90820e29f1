"""Walks of trees from two levels on, at the sizes where a level is added and
where walks of few rays change their starting level (3 to 7 levels), with few
rays per wavefront and with many, in both record forms, against the oracle bit
for bit."""
import numpy as np
import pytest

import vpo
from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walk", ["f16", "f32"])
@pytest.mark.parametrize("per_cu", [0, 1])
@pytest.mark.parametrize("n", [4, 16, 17, 64, 65, 1025, 16384, 16385])
def test_tree_depths_bitexact(ctx, n, per_cu, walk):
    rows = scenes.random_scene(n, 21, smin=0.4 / n ** 0.5, smax=1.2 / n ** 0.5, albedo=0.9, rho_scale=0.3 * n ** 0.25)
    env = scenes.sky_env(64, 32, sun_radius_deg=4.0, sun_scale=50.0)
    w, h, spp = 17, 9, 16 if per_cu and n < 2000 else 1
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    p = volprim.default_params(width=w, height=h, spp=spp, seed=5, max_depth=10, phase_g=0.2)
    print(f"[case] {n} Gaussians, {walk} records, {w}x{h}x{spp}", flush=True)
    sc, ev = ctx.scene(rows, bvh="median", walk=walk), ctx.env(env)
    _, _, rec, _ = sc.export()
    launch = volprim.LaunchConfig(64, per_cu, 0, 0, 0, volprim.PIPELINE_MEGAKERNEL, 0)
    img = ctx.render_jobs([(sc, ev, cam, p)], launch=launch)[0][0]
    sc.close()
    ev.close()
    ref, _, _ = vpo.render(rec, env, cam.pod(), w, h, spp, seed=5, max_depth=10, phase_g=0.2)
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
