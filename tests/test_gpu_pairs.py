"""The face-pair search at the edges of its clusters (64 leaves), groups and levels, against the oracle."""
import numpy as np
import pytest

import oracle
from collisiondetection_amd import api, scenes


def _loose_triangles(F, seed, size):
    """F triangles that share no vertex, at random places of the unit cube, each moving a little."""
    rng = np.random.default_rng(seed)
    q = rng.uniform(size=(F, 1, 3)) + rng.uniform(-size, size, size=(F, 3, 3))
    faces = np.arange(3 * F, dtype=np.int32).reshape(F, 3)
    return faces, q.reshape(-1, 3), (q + rng.normal(0.0, 0.3 * size, size=q.shape)).reshape(-1, 3)


def _check(faces, qs, qe, eta):
    vf, ee = api.kdop_candidates(faces, qs, qe, eta)
    ovf, oee = oracle.candidates(faces, oracle.Hist.two_entry(qs, qe), eta, method="tree")
    np.testing.assert_array_equal(vf, ovf)
    np.testing.assert_array_equal(ee, oee)
    return len(vf)


@pytest.mark.gpu
@pytest.mark.parametrize("F", [2, 63, 64, 65, 127, 128, 129, 4095, 4096, 4097])
def test_pairs_at_cluster_edges(F):
    n = _check(*_loose_triangles(F, F, 0.5 / F ** (1 / 3)), 1e-3)
    assert n > 0 or F == 2


@pytest.mark.gpu
@pytest.mark.parametrize("F", [2047, 2048, 2049, 262144, 262145])
def test_pairs_at_sort_tiles(F):
    """Around a sort tile (2,048 keys) and the most tiles that the scatter adds up by itself (128)."""
    assert _check(*_loose_triangles(F, F, 0.3 / F ** (1 / 3)), 1e-4) > 0


@pytest.mark.gpu
def test_pairs_all_overlapping():
    """Every leaf meets every other: full tiles, the output queue written several times."""
    faces, qs, qe = _loose_triangles(200, 1, 3.0)
    assert _check(faces, qs, qe, 1.0) > 100000


@pytest.mark.gpu
def test_pairs_flat_and_touching():
    """A lattice of squares in one plane: an axis without extent, and boxes that touch exactly."""
    v, f = scenes.grid(9)
    assert _check(f, v, v, 1.0 / 16.0) > _check(f, v, v, 1.0 / 16.0 - 1e-9)


@pytest.mark.gpu
def test_pairs_group_level():
    """More than 2048 clusters: the search scans groups of clusters."""
    s = scenes.cloth(n=264, noise=0.001)
    assert len(s["faces"]) > 2048 * 64
    assert _check(s["faces"], s["qstart"], s["qend"], s["eta"]) > 0


@pytest.mark.gpu
def test_pairs_third_level():
    """More than 2048 groups (8.4M faces): a lattice of far-apart small triangles with planted pairs."""
    n = 2048 * 64 * 64 + 3
    i = np.arange(n)
    c = np.stack([i % 256, i // 256 % 256, i // 65536], axis=1).astype(np.float64)
    corner = np.array([[0.0, 0.0, 0.0], [0.1, 0.0, 0.0], [0.0, 0.1, 0.05]])
    q = c[:, None, :] + corner[None]
    rng = np.random.default_rng(2)
    a = rng.choice(n // 2, size=500, replace=False)
    b = n // 2 + rng.choice(n // 2, size=500, replace=False)
    q[b] = q[a] + 0.01
    faces = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    vf, _ = api.kdop_candidates(faces, q, q, 1e-6)
    pairs = {(int(r[0]) // 3, int(r[1]) // 3) for r in vf}
    assert pairs == {(int(x), int(y)) for x, y in zip(a, b)} | {(int(y), int(x)) for x, y in zip(a, b)}


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[1, 2, 61, 3, 70, 64, 5, 128, 1, 40], [3] * 50])
def test_pairs_instances_within_a_cluster(sizes):
    """Instances that start and end inside a cluster overlap one another in space: no pair crosses them."""
    parts = [_loose_triangles(F, 10 + k, 0.2) for k, F in enumerate(sizes)]
    inst = [{"faces": f, "qstart": a, "qend": b} for f, a, b in parts]
    r = api.Batch(inst).detect(1e-3, 1e-3)
    nvf = nee = 0
    for f, a, b in parts:
        vf, ee = oracle.candidates(f, oracle.Hist.two_entry(a, b), 1e-3, method="tree")
        nvf, nee = nvf + len(vf), nee + len(ee)
    assert (r["vf_candidates"], r["ee_candidates"]) == (nvf, nee) and nvf > 0


@pytest.mark.gpu
@pytest.mark.parametrize("n,fins", [(9, False), (90, False), (150, False), (150, True)])
def test_stencils_of_a_face_over_many(n, fins):
    """A triangle whose swept bounds hold a whole lattice: its stencils with every vertex, edge and face of
    it, besides the lattice's own.  Its row has up to 793 clusters (more than the union's table holds);
    with fins there are edges of three faces."""
    v, f = scenes.grid(n)
    if fins:
        base = f[::7, :2]
        apex = v[base].mean(axis=1) + [0.0, 0.0, 1e-4]
        f = np.concatenate([f, np.column_stack([base, len(v) + np.arange(len(base))])]).astype(np.int32)
        v = np.concatenate([v, apex])
    eta = 1e-9
    own_vf, own_ee = api.kdop_candidates(f, v, v, eta)
    big, shift = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.0, 1.0, 1.0]]), np.array([50.0, 60.0, 70.0])
    nv = len(v)
    vf, ee = api.kdop_candidates(np.concatenate([f, [[nv, nv + 1, nv + 2]]]).astype(np.int32),
                                 np.concatenate([v, big - shift]), np.concatenate([v, big + shift]), eta)
    fs = np.sort(f, axis=1)
    edges = np.unique(np.sort(np.concatenate([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]]), axis=1), axis=0)
    want_vf = [own_vf, np.column_stack([np.arange(nv), np.tile([nv, nv + 1, nv + 2], (nv, 1))])]
    want_vf += [np.column_stack([np.full(len(fs), nv + k), fs]) for k in range(3)]
    want_ee = [own_ee] + [np.column_stack([edges, np.tile([nv + a, nv + b], (len(edges), 1))])
                          for a, b in ((0, 1), (0, 2), (1, 2))]
    np.testing.assert_array_equal(vf, np.unique(np.concatenate(want_vf), axis=0))
    np.testing.assert_array_equal(ee, np.unique(np.concatenate(want_ee), axis=0))
