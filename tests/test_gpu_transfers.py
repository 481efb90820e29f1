"""Copies between the host and the device around the slot size (1 MiB) and past
the eight slots: scene builds and exports, images, invalid input in a late
slot, and two threads on one context."""
import threading

import numpy as np
import pytest

import vpo
from volprim_amd import scenes, volprim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16384, 18724, 18725, 150000, 170000])
def test_build_and_export(ctx, n):
    rows = scenes.random_scene(n, 5)
    print(f"[case] build and export n={n}", flush=True)
    sc = ctx.scene(rows)
    got = [None, None]

    def export(k):
        got[k] = sc.export()

    threads = [threading.Thread(target=export, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    sc.close()
    codes = vpo.morton_codes(rows[:, 0:3])
    want = vpo.sort_order(codes)
    recs = vpo.make_prims(rows)[want].view(np.uint32)
    for order, morton, rec, _ in got:
        assert np.array_equal(morton, codes)
        assert np.array_equal(order, want)
        assert np.array_equal(rec.view(np.uint32), recs)


@pytest.mark.parametrize("bad", [[149999], [149000, 20000], [0]])
def test_invalid_primitive_is_named(ctx, bad):
    rows = scenes.random_scene(150000, 5)
    rows[bad, 9] = np.nan
    print(f"[case] invalid primitives {bad}", flush=True)
    with pytest.raises(Exception, match=f"primitive {min(bad)}: "):
        ctx.scene(rows)


@pytest.mark.parametrize("w,h", [(16, 4096), (16, 4097), (512, 1100)])
def test_images_match_device_output(ctx, w, h):
    torch = pytest.importorskip("torch")
    sc, ev = ctx.scene(scenes.random_scene(20, 2)), ctx.env(scenes.sky_env(16, 8, sun_radius_deg=4.0, sun_scale=50.0))
    cam = volprim.camera_perspective(**scenes.default_camera_args(w, h))
    p = volprim.default_params(width=w, height=h, spp=1, seed=3, max_depth=3)
    print(f"[case] image {w}x{h}", flush=True)
    dev = torch.empty((h, w, 4), dtype=torch.float32, device="cuda")
    ctx.render_device(sc, ev, cam, p, dev.data_ptr())
    want = dev.cpu().numpy().view(np.uint32)
    one = ctx.render(sc, ev, cam, p)[0]
    both = ctx.render_jobs([(sc, ev, cam, p)] * 2)[0]
    sc.close()
    ev.close()
    for img in [one, *both]:
        assert np.array_equal(np.asarray(img).view(np.uint32), want)
