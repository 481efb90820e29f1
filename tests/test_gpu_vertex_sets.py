"""The vertex stage's wave-wide passes over the active sets (rebuild, albedo,
chords from the vertex) at set sizes around the wavefront's 64 lanes, the four
entries read at a time and the longest list merged by scanning (1024), with
room for every member and with the set overflowing, against the oracle bit for
bit."""
import numpy as np
import pytest

import vpo
from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu


# n Gaussians that nearly all overlap: a path that scatters inside holds about
# n of them, most entered on one ray (1100: the lane-by-lane merge)
@pytest.mark.parametrize("ris", [0, 1])
@pytest.mark.parametrize("n,cap", [(1, 1), (3, 4), (5, 3), (63, 64), (64, 64), (65, 66), (130, 131), (130, 97),
                                   (1100, 1100), (1100, 1060)])
def test_overlapping_sets_bitexact(ctx, n, cap, ris):
    rows = scenes.random_scene(n, 11, extent=0.05, smin=0.15, smax=0.4, albedo=0.95, rho_scale=4.0 / n)
    env = scenes.sky_env(64, 32, sun_radius_deg=4.0, sun_scale=50.0)
    w, h, spp = 9, 8, 3
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    p = volprim.default_params(width=w, height=h, spp=spp, seed=9, max_depth=12, rr_depth=4, phase_g=0.4,
                               active_cap=cap, use_ris=ris)
    print(f"[case] {n} overlapping Gaussians, capacity {cap}, ris {ris}", flush=True)
    sc, ev = ctx.scene(rows), ctx.env(env)
    _, _, rec, _ = sc.export()
    img, st = ctx.render(sc, ev, cam, p)
    sc.close()
    ev.close()
    ref, _, k = vpo.render(rec, env, cam.pod(), w, h, spp, seed=9, max_depth=12, rr_depth=4, phase_g=0.4,
                           active_cap=cap, use_ris=bool(ris))
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
    assert st["active_overflow"] == k["active_overflow"]
