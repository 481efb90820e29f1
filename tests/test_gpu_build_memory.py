"""A scene built where the device has too little memory for all of the build's
temporaries at once (at 4^11 + 1 Gaussians 1.9 GB, and the scene's own 0.3 and
0.4), but enough for one stage after the other (1.5 GB with the scene): the
same order, codes, records and tree."""
import numpy as np
import pytest

from volprim_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walk,room", [("auto", 1800), ("auto", 2300), ("f32", 1800)])
def test_build_in_stages(ctx, walk, room):
    import torch
    n = 4 ** 11 + 1
    rng = np.random.default_rng(5)
    rows = np.empty((n, scenes.random_scene(4, 5).shape[1]), np.float32)
    rows[:] = scenes.random_scene(4, 5)[rng.integers(0, 4, n)]
    rows[:, 0:3] = rng.uniform(-1.0, 1.0, (n, 3))
    rows[:, 7:10] = rng.uniform(0.001, 0.004, (n, 3))
    rays = np.concatenate([np.full((64, 3), -2.0), rng.uniform(0.5, 1.5, (64, 3))], axis=1).astype(np.float32)

    def build():
        sc = ctx.scene(rows, walk=walk)
        out = *sc.export(), ctx.transmittance_rays(sc, rays), *sc.walk_info()
        sc.close()
        return out

    print(f"[case] {n} Gaussians, walk={walk}", flush=True)
    whole = build()
    torch.cuda.empty_cache()
    hog = []
    while (left := torch.cuda.mem_get_info()[0] - room * 10 ** 6) > 1 << 26:
        hog.append(torch.empty(min(left, 16 << 30), dtype=torch.uint8, device="cuda"))
    print(f"[case] the same with {torch.cuda.mem_get_info()[0] // 10 ** 6} MB free", flush=True)
    try:
        staged = build()
    finally:
        del hog
        torch.cuda.empty_cache()
    for a, b in zip(whole[:-1], staged[:-1]):
        assert np.asarray(a).tobytes() == np.asarray(b).tobytes()
    assert abs(whole[-1] - staged[-1]) < 1e-9  # the tree's growth: a sum in no fixed order
