"""Scene builds at the sizes where the sort takes another tile, its histogram
scan another round and the bounds fold another partial, and with many equal
Morton codes: order, codes, records and tree depth against the CPU."""
import numpy as np
import pytest

import vpo
from volprim_amd import scenes

pytestmark = pytest.mark.gpu


def radix_depth(codes):
    """Depth of the binary radix tree over sorted 32-bit codes, ties by index."""
    keys = (codes.astype(np.uint64) << np.uint64(32)) | np.arange(len(codes), dtype=np.uint64)
    depth, todo = 0, [(0, len(keys), 0)]
    while todo:
        lo, hi, d = todo.pop()
        depth = max(depth, d)
        if hi - lo < 2:
            continue
        bit = int(keys[lo] ^ keys[hi - 1]).bit_length() - 1
        split = (int(keys[hi - 1]) >> bit) << bit
        mid = lo + int(np.searchsorted(keys[lo:hi], np.uint64(split)))
        todo += [(lo, mid, d + 1), (mid, hi, d + 1)]
    return depth


@pytest.mark.parametrize("same", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 65, 256, 257, 2048, 2049, 16640, 65536, 65537])
def test_build_sizes(ctx, n, same):
    rows = scenes.random_scene(n, 3)
    if same:
        rows[:, 0:3] = rows[: min(n, 5), 0:3][np.arange(n) % min(n, 5)]
    print(f"[case] scene build n={n} same={same}", flush=True)
    sc = ctx.scene(rows)
    order, morton, rec, depth = sc.export()
    sc.close()
    codes = vpo.morton_codes(rows[:, 0:3])
    assert np.array_equal(morton, codes)
    assert np.array_equal(order, vpo.sort_order(codes))
    assert np.array_equal(rec.view(np.uint32), vpo.make_prims(rows)[order].view(np.uint32))
    assert depth == radix_depth(codes[order])
