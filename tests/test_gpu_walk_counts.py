"""Walk counts of the counting build against their exact values: in a scene of
n concentric, equal Gaussians a ray that crosses one leaf box crosses all of
them and every node's box above, so per ray there is the root, and per crossing
ray every other node that has leaves, and n leaf tests."""
import numpy as np
import pytest

from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walk", ["f16", "f32"])
@pytest.mark.parametrize("n", [1, 4, 5, 16, 17, 50])
def test_concentric_walk_counts(ctx, n, walk):
    rows = np.repeat(scenes.c0_single_gaussian(), n, axis=0)
    rows[:, 10:13] = 0.8
    rows[:, 13] /= n
    w, h = 24, 16
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    p = volprim.default_params(width=w, height=h, spp=4, seed=3, phase_g=0.3, max_depth=8)
    print(f"[case] {n} concentric Gaussians, {walk}", flush=True)
    sc, ev = ctx.scene(rows, walk=walk), ctx.env(scenes.sky_env(32, 16, sun_radius_deg=4.0, sun_scale=50.0))
    e = ctx.count_events(sc, ev, cam, p)
    sc.close()
    ev.close()
    rays = e["traces"] + e["shadow_rays"]
    nodes = -(-n // 4) + (-(-n // 16) if n > 16 else 0)  # below the root
    assert e["leaf_tests"] > 0 and e["leaf_tests"] % n == 0
    crossing = e["leaf_tests"] // n
    assert e["node_visits"] - e["visits_point"] == rays + nodes * crossing
