"""Active sets of more than a thousand members, most of them entered on one ray,
with room for all and with the set overflowing, against the oracle bit for
bit."""
import numpy as np
import pytest

import vpo
from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cap", [(1025, 1025), (2100, 2100), (2100, 1700)])
def test_large_sets_bitexact(ctx, n, cap):
    rows = scenes.random_scene(n, 11, extent=0.05, smin=0.15, smax=0.4, albedo=0.95, rho_scale=4.0 / n)
    env = scenes.sky_env(64, 32, sun_radius_deg=4.0, sun_scale=50.0)
    w, h = 9, 8
    kw = dict(seed=9, max_depth=8, rr_depth=4, phase_g=0.4, active_cap=cap)
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    print(f"[case] {n} overlapping Gaussians, capacity {cap}", flush=True)
    sc, ev = ctx.scene(rows), ctx.env(env)
    _, _, rec, _ = sc.export()
    img, st = ctx.render(sc, ev, cam, volprim.default_params(width=w, height=h, spp=2, **kw))
    sc.close()
    ev.close()
    ref, _, k = vpo.render(rec, env, cam.pod(), w, h, 2, **kw)
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
    assert st["active_overflow"] == k["active_overflow"]
