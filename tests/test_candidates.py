"""Candidate generation: ori_local_sampling.m and find_neighbor_ORs.m."""
import ctypes

import numpy as np
import pytest

import oracle

EPS = np.finfo(float).eps


# -- the colon operator (MathWorks' published examples of a:d:b) -------------

def test_colon_documented_examples():
    # 1-eps : eps/4 : 1+eps is the nine doubles nearest 1 + (-4:4)*eps/4
    v = oracle.colon(1 - EPS, EPS / 4, 1 + EPS)
    np.testing.assert_array_equal(v, [1 - EPS, 1 - EPS, 1 - EPS / 2, 1, 1, 1, 1, 1 + EPS, 1 + EPS])
    # -1 : 0.01 : 1 is 201 values symmetric about an exact zero
    v = oracle.colon(-1.0, 0.01, 1.0)
    assert v.size == 201 and v[100] == 0.0
    np.testing.assert_array_equal(v, -v[::-1])


def test_colon_integer_and_empty_cases():
    np.testing.assert_array_equal(oracle.colon(1, 1, 5), [1, 2, 3, 4, 5])
    np.testing.assert_array_equal(oracle.colon(10, -3, 1), [10, 7, 4, 1])
    np.testing.assert_array_equal(oracle.colon(0.5, 1, 3.2), [0.5, 1.5, 2.5])
    assert oracle.colon(1, 1, 0).size == 0
    assert oracle.colon(1, 0, 5).size == 0
    assert oracle.colon(1, -1, 5).size == 0


def test_colon_grid_of_local_sampling():
    c, g, nr = 0.1234567, 0.004, 8
    v = oracle.colon(c - (g * nr) / 2, g, c + (g * nr) / 2)
    assert v.size == nr + 1
    assert v[0] == c - (g * nr) / 2 and v[-1] == c + (g * nr) / 2   # both ends exact
    np.testing.assert_allclose(np.diff(v), g, rtol=1e-12)


# -- ori_local_sampling -------------------------------------------------------

def _rows_numpy(centre, nr, g):
    """Independent restatement: rows in loop order, then numpy's lexicographic unique."""
    half = (g * nr) / 2
    grids = [oracle.colon(centre[j] - half, g, centre[j] + half) for j in (1, 2, 3)]
    rows = [np.asarray(centre, float)]
    for b in grids[0]:
        for c in grids[1]:
            for d in grids[2]:
                rows.append([np.sqrt(1 - ((b * b + c * c) + d * d)), b, c, d])
    return np.unique(np.array(rows), axis=0)


@pytest.mark.parametrize("nr,g", [(8, 0.004), (4, 0.004), (5, 0.004), (6, 0.0043633)])
def test_local_sampling_matches_numpy_unique(nr, g):
    rng = np.random.default_rng(nr)
    for _ in range(4):
        v = rng.normal(size=3)
        v *= rng.uniform(0.05, 0.4) / np.linalg.norm(v)
        centre = np.array([np.sqrt(1 - v @ v), *v])
        q = oracle.local_sampling(centre, nr, g)
        np.testing.assert_array_equal(q, _rows_numpy(centre, nr, g))
        assert q.shape[0] in ((nr + 1) ** 3, (nr + 1) ** 3 + 1)


def test_local_sampling_centre_survives_only_when_distinct():
    # a centre that equals its grid's middle point merges (729 rows); a q0
    # off in the last bit keeps the prepended centre (730 rows)
    g, nr = 0.004, 8
    half = (g * nr) / 2
    c = np.array([0.0, 0.125, -0.25, 0.0625])   # dyadic: the middle grid value is exact
    mids = [oracle.colon(x - half, g, x + half)[nr // 2] for x in c[1:]]
    assert mids == list(c[1:])
    c[0] = np.sqrt(1 - ((c[1] * c[1] + c[2] * c[2]) + c[3] * c[3]))
    assert oracle.local_sampling(c, nr, g).shape[0] == 729
    c2 = c.copy()
    c2[0] = np.nextafter(c[0], 2.0)
    q = oracle.local_sampling(c2, nr, g)
    assert q.shape[0] == 730
    assert (q == c2).all(axis=1).sum() == 1


def test_local_sampling_rows_sorted_and_unit():
    q = oracle.local_sampling([0.05, 0.1, -0.2], 8, 0.004)   # 3-vector centre: q0 recomputed
    assert np.all(np.diff(q[:, 0]) >= 0)
    order = np.lexsort(q.T[::-1])
    np.testing.assert_array_equal(order, np.arange(q.shape[0]))
    np.testing.assert_allclose(np.sum(q * q, axis=1), 1.0, atol=1e-15)


# -- find_neighbor_ORs ---------------------------------------------------------

def _neighbors_numpy(gid, vox, radius, nr_max):
    dims = gid.shape
    ids, ind = [], []
    for p in vox:
        r = radius
        while True:
            lo = [max(p[j] - r, 1) if p[j] - r > 0 else 1 for j in range(3)]
            hi = [p[j] + r if p[j] + r < dims[j] else dims[j] for j in range(3)]
            box = gid[lo[0] - 1:hi[0], lo[1] - 1:hi[1], lo[2] - 1:hi[2]]
            u = np.unique(box[box > 0])
            if u.size:
                break
            r += 2
        u = u[:nr_max]
        ind.append([len(ids) + 1, len(ids) + u.size])
        ids.extend(u.tolist())
    return np.array(ids, np.int32), np.array(ind, np.int64)


def _volume(rng, shape, fill, ngrains):
    gid = np.zeros(shape, np.int32)
    mask = rng.random(shape) < fill
    gid[mask] = rng.integers(1, ngrains + 1, size=mask.sum())
    return gid


@pytest.mark.parametrize("fill,radius,nr_max", [(0.3, 2, 30), (0.002, 1, 30), (0.5, 3, 5)])
def test_find_neighbor_ors_matches_numpy(fill, radius, nr_max):
    rng = np.random.default_rng(int(fill * 1000) + radius)
    gid = _volume(rng, (17, 13, 11), fill, 120)
    vox = np.stack([rng.integers(1, n + 1, 40) for n in gid.shape], axis=1)
    ids, ind = oracle.find_neighbor_ors(gid, vox, radius, nr_max)
    ids2, ind2 = _neighbors_numpy(gid, vox, radius, nr_max)
    np.testing.assert_array_equal(ids, ids2)
    np.testing.assert_array_equal(ind, ind2)


def test_find_neighbor_ors_empty_volume_is_an_error():
    with pytest.raises(ValueError):
        oracle.find_neighbor_ors(np.zeros((4, 4, 4), np.int32), [[1, 1, 1]], 1)


# -- the engine ----------------------------------------------------------------

@pytest.mark.gpu
def test_engine_local_sampling_matches_oracle(engine):
    rng = np.random.default_rng(5)
    cs = []
    for _ in range(24):
        v = rng.normal(size=3)
        v *= rng.uniform(0.01, 0.45) / np.linalg.norm(v)
        cs.append([np.sqrt(1 - v @ v), *v])
    cs.append([0.0, 0.125, -0.25, 0.0625])
    cs[-1][0] = np.sqrt(1 - ((0.125 * 0.125 + 0.25 * 0.25) + 0.0625 * 0.0625))
    cs = np.array(cs)
    for nr, g in [(8, 0.004), (4, 0.004), (6, 0.0043633), (10, 0.001)]:
        got = engine.local_sampling(cs, nr, g)
        for k in range(cs.shape[0]):
            np.testing.assert_array_equal(got[k], oracle.local_sampling(cs[k], nr, g))


@pytest.mark.gpu
def test_engine_find_neighbor_ors_matches_oracle(engine):
    rng = np.random.default_rng(9)
    for fill, radius, nr_max, ng in [(0.3, 3, 30, 300), (0.001, 2, 30, 50), (0.6, 4, 7, 2000)]:
        gid = _volume(rng, (40, 33, 29), fill, ng)
        vox = np.stack([rng.integers(1, n + 1, 500) for n in gid.shape], axis=1)
        ids, ind = engine.find_neighbor_ors(gid, vox, radius, nr_max)
        ids2, ind2 = oracle.find_neighbor_ors(gid, vox, radius, nr_max)
        np.testing.assert_array_equal(ids, ids2)
        np.testing.assert_array_equal(ind, ind2)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 4228, 4229])
def test_engine_find_neighbor_ors_list_sizes(engine, M):
    """Lists packed by the host (up to 512 KB: 4,228 voxels of 30 ids and a
    count) and on the device; the caller's memory behind the ids stays as it
    was."""
    rng = np.random.default_rng(M)
    gid = _volume(rng, (30, 23, 19), 0.05, 400)
    vox = np.stack([rng.integers(1, n + 1, M) for n in gid.shape], axis=1)
    want = oracle.find_neighbor_ors(gid, vox, 3, 30)
    for a, b in zip(engine.find_neighbor_ors(gid, vox, 3), want):
        np.testing.assert_array_equal(a, b)
    ids, ind, n = np.full(30 * M, -7, np.int32), np.zeros((M, 2), np.int64), ctypes.c_int64()
    flat, v = np.ascontiguousarray(gid.reshape(-1, order="F")), np.ascontiguousarray(vox, dtype=np.int32)
    p = lambda a: a.ctypes.data_as(ctypes.POINTER(np.ctypeslib.as_ctypes_type(a.dtype)))  # noqa: E731
    engine._chk(engine._lib.grs_find_neighbor_ors(engine._h, p(flat), *gid.shape, p(v), M, 3, 30, p(ids), p(ind),
                                                  ctypes.byref(n)))
    assert n.value == want[0].size and np.array_equal(ids[:n.value], want[0]) and (ids[n.value:] == -7).all()
    np.testing.assert_array_equal(ind, want[1])


@pytest.mark.gpu
def test_engine_candidate_errors(engine):
    from grainrecon_amd._lib import GrsError

    with pytest.raises(GrsError):
        engine.find_neighbor_ors(np.zeros((4, 4, 4), np.int32), np.array([[1, 1, 1]]), 1)
    with pytest.raises(GrsError):
        engine.find_neighbor_ors(np.ones((4, 4, 4), np.int32), np.array([[5, 1, 1]]), 1)
    with pytest.raises(GrsError):
        engine.local_sampling([0.9, 0.1, 0.2, 0.3], 20, 0.004)   # 9262 rows > 2048
