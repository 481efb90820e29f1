"""Walks shared between the wavefronts of a workgroup: scenes whose walks have
more items than one wavefront takes at once, at the path counts where
workgroups grow (16 and 32 paths to a compute unit of 256), one scene and
wavefronts over two, against the oracle bit for bit."""
import numpy as np
import pytest

import vpo
from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu


def dense(n, seed):
    return scenes.random_scene(n, seed, smin=0.05, smax=0.3, albedo=0.95, rho_scale=40.0 / n)


@pytest.mark.parametrize("ris", [False, True])
@pytest.mark.parametrize("w,h", [(8, 8), (64, 63), (64, 64), (64, 127), (64, 128), (96, 160)])
def test_helped_walks_bitexact(ctx, w, h, ris):
    env = scenes.sky_env(32, 16, sun_radius_deg=4.0, sun_scale=50.0)
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    p = volprim.default_params(width=w, height=h, spp=1, seed=9, max_depth=24, phase_g=0.5, use_ris=int(ris))
    print(f"[case] 1500 Gaussians, {w}x{h}, ris={ris}", flush=True)
    sc, ev = ctx.scene(dense(1500, 31), bvh="median"), ctx.env(env)
    _, _, rec, _ = sc.export()
    img = ctx.render(sc, ev, cam, p)[0]
    sc.close()
    ev.close()
    ref, _, _ = vpo.render(rec, env, cam.pod(), w, h, 1, seed=9, max_depth=24, phase_g=0.5, use_ris=int(ris))
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))


def test_helped_walks_over_two_scenes(ctx):
    env = scenes.sky_env(32, 16, sun_radius_deg=4.0, sun_scale=50.0)
    w, h = 8, 8
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    p = volprim.default_params(width=w, height=h, spp=3, seed=9, max_depth=16, phase_g=0.5)
    print("[case] 120 jobs over two scenes", flush=True)
    scs, ev = [ctx.scene(dense(n, 31), bvh="median") for n in (900, 1500)], ctx.env(env)
    recs = [sc.export()[2] for sc in scs]
    imgs = ctx.render_jobs([(scs[k % 2], ev, cam, p) for k in range(120)])[0]
    for sc in scs:
        sc.close()
    ev.close()
    refs = [vpo.render(rec, env, cam.pod(), w, h, 3, seed=9, max_depth=16, phase_g=0.5)[0] for rec in recs]
    for k, img in enumerate(imgs):
        assert np.array_equal(img.view(np.uint32), refs[k % 2].view(np.uint32)), k
