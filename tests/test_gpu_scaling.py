"""Calls whose time must not grow faster than their input: device times of a stage at two sizes."""
import ctypes

import numpy as np
import pytest

from collisiondetection_amd import _native as N
from collisiondetection_amd import api, scenes

pytestmark = pytest.mark.gpu


def _stage_ms(ctx, stage, call):
    """The least time of a stage over three calls."""
    L = N.lib()
    ms, calls = (ctypes.c_double * N.NTIMERS)(), (ctypes.c_int64 * N.NTIMERS)()
    best = np.inf
    call()
    L.ccd_set_profiling(ctx.ptr, 1)
    for _ in range(3):
        L.ccd_stage_times(ctx.ptr, None, None, 1)
        call()
        L.ccd_stage_times(ctx.ptr, ms, calls, 1)
        best = min(best, ms[stage])
    L.ccd_set_profiling(ctx.ptr, 0)
    return best


def test_expansion_over_a_ground_of_two_triangles():
    """A cloth over two large triangles that its every face meets: four times the faces, and four times the
    work, take well below the sixteen times and more of a search in the large triangles' rows."""
    ctx = api.Context()
    times = []
    for n in (150, 300):
        s = scenes.cloth(n)
        nv = len(s["qstart"])
        q = np.array([[-1.0, -1.0, -0.2], [3.0, -1.0, -0.2], [-1.0, 3.0, -0.2], [3.0, 3.0, -0.2]])
        faces = np.concatenate([s["faces"], [[nv, nv + 1, nv + 2], [nv + 1, nv + 3, nv + 2]]]).astype(np.int32)
        qs, qe = np.concatenate([s["qstart"], q]), np.concatenate([s["qend"], q + [0.0, 0.0, 0.5]])
        times.append(_stage_ms(ctx, N.TIMER_NAMES.index("expand"), lambda: api.kdop_candidates(faces, qs, qe, 1e-6, sort=False, ctx=ctx)))
        print("case: ground under a cloth", n, "expansion ms", times[-1], flush=True)
    assert times[1] < 12.0 * times[0]


def test_search_with_a_body_far_away():
    """A sheet whose faces are in no order, and with a triangle 10^5 times its size away.  21 bits per axis leave
    the sheet 21 cells along each side: 18 clusters of faces in each, instead of one, at the places of the 9
    around it.  A search that finds no order in the sheet meets all 8,160 clusters for each."""
    ctx = api.Context()
    s = scenes.crumpled_sheet(512)
    faces = np.random.default_rng(1).permutation(s["faces"]).astype(np.int32)
    nv = len(s["qstart"])
    far = 1e5 * np.ones(3) + np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.0, 1.0, 0.0]])
    times = []
    for f, extra in ((faces, far[:0]), (np.concatenate([faces, [[nv, nv + 1, nv + 2]]]).astype(np.int32), far)):
        qs, qe = np.concatenate([s["qstart"], extra]), np.concatenate([s["qend"], extra])
        times.append(_stage_ms(ctx, N.TIMER_NAMES.index("traverse"),
                               lambda: api.kdop_candidates(f, qs, qe, 1e-7, sort=False, as_numpy=False, ctx=ctx)))
        print("case: a shuffled sheet,", len(extra) // 3, "bodies far away, search ms", times[-1], flush=True)
    assert times[1] < 60.0 * times[0]


def test_histories_that_nearly_all_collide():
    """Stencils that are closer than the thickness all the time take no more than a few times what those take that
    hardly ever are: their first windows decide them."""
    import time

    import torch

    rng = np.random.default_rng(3)
    V, entries, n = 40, 60, 8600
    t = [np.concatenate([[0], np.sort(rng.choice(np.arange(1, 1024), size=entries - 2, replace=False)), [1024]]) for _ in range(V)]
    hist = [np.arange(V + 1, dtype=np.int64) * entries, np.concatenate(t) / 1024.0,
            np.repeat(rng.uniform(size=(V, 3)), entries, axis=0) + rng.normal(0.0, 0.005, size=(V * entries, 3))]
    keys = np.stack([rng.permutation(V)[:4] for _ in range(n)]).astype(np.int32)
    args = [torch.from_numpy(a).cuda() for a in (*hist, keys, keys)]
    times, hits = [], []
    for eta in (1e-6, 2.0):
        best = np.inf
        for _ in range(4):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            r = api.narrowphase_history(*args, eta)
            best = min(best, time.perf_counter() - t0)
        times.append(best)
        hits.append(r["vf_hit"].mean())
        print("case: histories, thickness", eta, "ms", 1e3 * best, "collide", hits[-1], flush=True)
    assert hits[0] < 0.05 and hits[1] > 0.95 and times[1] < 4.0 * times[0]


def test_expansion_of_a_mesh_with_a_degenerate_face():
    """One degenerate face sends the whole mesh to the raw emission: fifteen stencils of every pair instead of each
    stencil once, a few times the keys, and no more than ten times the time."""
    ctx = api.Context()
    s = scenes.cloth(256)
    times = []
    for faces in (s["faces"], np.concatenate([s["faces"], [[0, 0, 1]]]).astype(np.int32)):
        times.append(_stage_ms(ctx, N.TIMER_NAMES.index("expand"),
                               lambda: api.kdop_candidates(faces, s["qstart"], s["qend"], s["eta"], sort=False, as_numpy=False,
                                                           ctx=ctx)))
        print("case: cloth with", len(faces) - len(s["faces"]), "degenerate faces, expansion ms", times[-1], flush=True)
    assert times[1] < 10.0 * times[0]


def test_one_pass_narrowphase_of_a_short_list():
    """87,000 edge-edge stencils in one pass with the solver, on all wavefronts: no more than four times the three
    passes, which run the solver on a tenth of them."""
    s = scenes.cloth(97)
    times = []
    for on in (True, False):
        ctx = api.Context()
        api.set_edge_edge_split(on, ctx)
        times.append(_stage_ms(ctx, N.TIMER_NAMES.index("narrow_ee"),
                               lambda: api.detect(s["faces"], s["qstart"], s["qend"], s["eta"], s["eta"], ctx=ctx)))
        print("case: edge-edge narrowphase,", "three passes" if on else "one pass", "ms", times[-1], flush=True)
    assert times[1] < 4.0 * times[0]
