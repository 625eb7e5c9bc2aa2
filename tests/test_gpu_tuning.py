"""Tuning times what the kernels depend on, and a stored shape belongs to the kernels it was tuned for."""
import json

import pytest

from collisiondetection_amd import api, scenes

pytestmark = pytest.mark.gpu


def test_only_the_tile_is_tuned():
    """The screening form reads no block size and no number of wavefronts: timer noise must not choose them."""
    ctx = api.Context()
    s = scenes.cloth(64, drop=0.05)
    shapes = []
    for _ in range(6):
        api.detect(s["faces"], s["qstart"], s["qend"], s["eta"], s["eta"], ctx=ctx)
        shapes.append(api.autotune(s["qstart"], s["qend"], s["eta"], ctx=ctx))
    assert len({(x[0], x[2], x[3], x[5]) for x in shapes}) == 1
    assert all(x[k] in (64, 128, 256, 512, 1024, 2048, 4096) for x in shapes for k in (1, 4))


def test_shape_stored_for_other_kernels(tmp_path):
    cache = str(tmp_path / "shapes.json")
    b = api.Batch(scenes.batched_instances(count=3, seed=7, tri_lo=200, tri_hi=800))
    assert b.tune(1e-6, 1e-6, cache=cache)[1] == "tuned"
    assert b.tune(1e-6, 1e-6, cache=cache)[1] == "cache"
    with open(cache) as fh:
        (key, shape), = json.load(fh).items()
    with open(cache, "w") as fh:   # as one without the kernels' name was stored
        json.dump({key[key.index("gfx"):]: shape}, fh)
    assert b.tune(1e-6, 1e-6, cache=cache)[1] == "tuned"
