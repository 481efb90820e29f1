"""Walks shared between the wavefronts of a workgroup in the forms that end or
record them otherwise: a scene whose walks have more items than one wavefront
takes at once, a tile row below and at the path counts where workgroups grow
(4096 and 8192 paths).  Images, and the measuring build's largest entry count
of a ray and largest overlap of a vertex, against the oracle."""
import numpy as np
import pytest

import vpo
from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu


def dense(n, seed):
    return scenes.random_scene(n, seed, smin=0.05, smax=0.3, albedo=0.95, rho_scale=40.0 / n)


@pytest.mark.parametrize("w,h", [(8, 8), (64, 56), (64, 64), (64, 120), (64, 128)])
def test_helped_measuring_walks(ctx, w, h):
    env = scenes.sky_env(32, 16, sun_radius_deg=4.0, sun_scale=50.0)
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    kw = dict(seed=9, max_depth=24, phase_g=0.5)
    print(f"[case] measuring, 1500 Gaussians, {w}x{h}", flush=True)
    sc, ev = ctx.scene(dense(1500, 31), bvh="median"), ctx.env(env)
    _, _, rec, _ = sc.export()
    img, st = ctx.render(sc, ev, cam, volprim.default_params(width=w, height=h, spp=1, measure_caps=1, **kw))
    sc.close()
    ev.close()
    ref, _, k = vpo.render(rec, env, cam.pod(), w, h, 1, measure=True, use_ris=False, **kw)
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
    assert st["max_hits_per_ray"] == k["max_hits"] and st["max_point_overlap"] == k["max_overlap"]


@pytest.mark.parametrize("w,h", [(64, 56), (64, 64), (64, 120), (64, 128)])
@pytest.mark.parametrize("form", ["roulette", "small_cap", "f32"])
def test_helped_walk_forms(ctx, form, w, h):
    # rays that end at a roulette's depth (two thirds of the pixels differ from the
    # image without it); more candidates than the capacity
    # (rebuilt by a point query); binary32 records
    env = scenes.sky_env(32, 16, sun_radius_deg=4.0, sun_scale=50.0)
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    kw = dict(seed=9, max_depth=24, phase_g=0.5)
    kw.update({"roulette": dict(shadow_rr=0.5), "small_cap": dict(active_cap=24), "f32": {}}[form])
    print(f"[case] {form}, 1500 Gaussians, {w}x{h}", flush=True)
    sc = ctx.scene(dense(1500, 31), bvh="median", walk="f32" if form == "f32" else "auto")
    ev = ctx.env(env)
    _, _, rec, _ = sc.export()
    img = ctx.render(sc, ev, cam, volprim.default_params(width=w, height=h, spp=1, **kw))[0]
    sc.close()
    ev.close()
    ref = vpo.render(rec, env, cam.pod(), w, h, 1, **kw)[0]
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
