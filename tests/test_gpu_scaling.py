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
