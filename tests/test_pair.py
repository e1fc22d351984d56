"""Spot pairing (forward_comp_pair_spots.m:3-93): the oracle pinned on
constructed spot lists, the GPU (grs_pair_spots) against the oracle."""
import ctypes

import numpy as np
import pytest

import oracle
import scenes
from oracle.pair_spots import pair_spots


@pytest.fixture(scope="module")
def scene():
    return scenes.make_scene(seed=83, ngrains=3, spread_mm=0.05, nrot=37)


def _frames_at_events(s, ev, offset=(0.0, 0.0), area=4.0):
    frames = [[] for _ in range(s.rot.size)]
    for om, _h, dy, dz, *_ in ev:
        frames[int(om)].append([dy + offset[0], dz + offset[1], area])
    return [np.array(f).reshape(-1, 3) for f in frames]


def test_oracle_pairing_known_answers(scene):
    s = scene
    U, p = s.U[0], s.centers[0]
    ns, ni, med, ev = oracle.forward_comp(s.geo, s.stack, U, p, s.rot, s.hkl, events=True)
    thr = s.geo.minEucDis / ((s.geo.pixelysize + s.geo.pixelzsize) / 2.0)
    hits = ev[ev[:, 6] <= thr]
    assert ni == hits.shape[0] > 20
    # a spot on every event pixel: every hit pairs at distance 0
    _, _, _, rows = pair_spots(s.geo, s.stack, U, p, s.rot, s.hkl, _frames_at_events(s, ev))
    assert rows.shape == (hits.shape[0], 23)
    np.testing.assert_array_equal(rows[:, 17:19], rows[:, 20:22])
    np.testing.assert_array_equal(rows[:, 20:22], hits[:, 2:4])
    np.testing.assert_array_equal(rows[:, 0:9], np.float32(U.flatten(order="F")).astype(float)[None, :].repeat(len(rows), 0))
    np.testing.assert_allclose(rows[:, 10], np.float32(p[1] - s.geo.RotAxisOffset))
    # Energy from the wavelength of each event (keV, 12.398/lambda in single precision)
    np.testing.assert_array_equal(rows[:, 15], np.float32(12.398 / hits[:, 7]).astype(float))
    # spots 5 px away: paired when sqrt(area) > 5, not when sqrt(area) = 4 or the distance reaches 15
    _, _, _, r36 = pair_spots(s.geo, s.stack, U, p, s.rot, s.hkl, _frames_at_events(s, ev, (3.0, 4.0), 36.0))
    _, _, _, r16 = pair_spots(s.geo, s.stack, U, p, s.rot, s.hkl, _frames_at_events(s, ev, (3.0, 4.0), 16.0))
    _, _, _, rfar = pair_spots(s.geo, s.stack, U, p, s.rot, s.hkl, _frames_at_events(s, ev, (9.0, 12.0), 900.0))
    assert r36.shape[0] == hits.shape[0] and r16.shape[0] == 0 and rfar.shape[0] == 0


def _frames(s, rng):
    """Spots near the events of every grain centre plus random ones."""
    frames = [[] for _ in range(s.rot.size)]
    for g in range(len(s.U)):
        _, _, _, ev = oracle.forward_comp(s.geo, s.stack, s.U[g], s.centers[g], s.rot, s.hkl, events=True)
        for om, _h, dy, dz, *_ in ev:
            frames[int(om)].append([dy + rng.uniform(-3, 3), dz + rng.uniform(-3, 3), rng.uniform(1, 60)])
    det = int(s.geo.detysize)
    for f in frames:
        for _ in range(int(rng.integers(0, 6))):
            f.append([rng.uniform(1, det), rng.uniform(1, det), rng.uniform(1, 400)])
    frames[3] = []  # a projection without spots
    return [np.array(f).reshape(-1, 3) for f in frames]


@pytest.mark.gpu
def test_pair_spots_equals_oracle(engine, scene):
    s = scene
    engine.set_geometry(s.geo, s.hkl, s.rot)
    engine.set_distance_stack(s.proj)
    rng = np.random.default_rng(11)
    frames = _frames(s, rng)
    engine.set_frame_spots(frames)
    pos = np.array([s.centers[0], s.centers[1], s.voxels[2][3], s.centers[2]])
    U = np.stack([s.U[0], s.U[1], s.U[2], scenes.U_from_qvec(*(s.q[2, 1:] + 0.004))])
    print(f"pair_spots: {pos.shape[0]} orientations, {sum(len(f) for f in frames)} spots", flush=True)
    ns, ni, med, rows = engine.pair_spots(pos, U)
    total = 0
    for m in range(pos.shape[0]):
        rns, rni, rmed, rrows = pair_spots(s.geo, s.stack, U[m], pos[m], s.rot, s.hkl, frames)
        assert (ns[m], ni[m], med[m]) == (rns, rni, np.float32(rmed)), m
        assert rows[m].shape == rrows.shape, m
        np.testing.assert_array_equal(rows[m], rrows)
        total += rrows.shape[0]
    assert total > 50


@pytest.mark.gpu
@pytest.mark.parametrize("per_frame, repeat", [(0, 1), (1, 1), (63, 1), (65, 1), (700, 1), (40, 40)])
def test_pair_spots_list_lengths(engine, scene, per_frame, repeat):
    """Projections without spots, with less and more than a wave reads at a
    time, spots repeated (the first one counts) or without a position (NaN),
    every selected event a hit; reflections repeated."""
    s = scene
    hkl = np.concatenate([s.hkl[:min(len(s.hkl), 240 // repeat)]] * repeat) if repeat > 1 else s.hkl
    engine.set_geometry(s.geo, hkl, s.rot)
    proj = np.zeros_like(s.proj)
    engine.set_distance_stack(proj)
    import oracle

    stack = oracle.Stack(proj)
    rng = np.random.default_rng(per_frame + repeat)
    _, _, _, ev = oracle.forward_comp(s.geo, stack, s.U[0], s.centers[0], s.rot, hkl, events=True)
    frames = [[] for _ in range(s.rot.size)]
    for e in ev:
        if per_frame and len(frames[int(e[0])]) < per_frame:
            frames[int(e[0])].append([e[2] + rng.uniform(-3, 3), e[3] + rng.uniform(-3, 3), rng.uniform(1, 300)])
    det = float(s.geo.detysize)
    full = []
    for f in frames:
        f = np.array(f, float).reshape(-1, 3)
        f = np.concatenate([f, f[:per_frame // 3]])[:per_frame]
        more = np.column_stack([rng.uniform(1, det, (per_frame - len(f), 2)), np.full(per_frame - len(f), 100.0)])
        f = np.concatenate([f, more])
        if len(f) > 2:
            f[1, 0] = np.nan
        full.append(f)
    engine.set_frame_spots(full)
    ns, ni, med, rows = engine.pair_spots(s.centers[:1], s.U[0][None])
    rns, rni, rmed, rrows = pair_spots(s.geo, stack, s.U[0], s.centers[0], s.rot, hkl, full)
    assert (ns[0], ni[0], med[0]) == (rns, rni, np.float32(rmed))
    np.testing.assert_array_equal(rows[0], rrows.reshape(-1, 23))


@pytest.mark.gpu
def test_pair_spots_of_more_rows_than_the_first_call_holds(engine):
    """A dense set of events (181 angles, 240 reflections, every selected
    event a hit with a spot of its own) pairs more than 1024 spots."""
    import oracle

    s = scenes.make_scene(seed=84, ngrains=1, spread_mm=0.02, nrot=181)
    hkl = np.concatenate([s.hkl, s.hkl, s.hkl])[:240]
    proj = np.zeros_like(s.proj)
    engine.set_geometry(s.geo, hkl, s.rot)
    engine.set_distance_stack(proj)
    stack = oracle.Stack(proj)
    _, _, _, ev = oracle.forward_comp(s.geo, stack, s.U[0], s.centers[0], s.rot, hkl, events=True)
    assert len(ev) > 1024
    frames = _frames_at_events(s, ev)
    engine.set_frame_spots(frames)
    ns, ni, med, rows = engine.pair_spots(s.centers[:1], s.U[0][None])
    rns, rni, rmed, rrows = pair_spots(s.geo, stack, s.U[0], s.centers[0], s.rot, hkl, frames)
    assert rows[0].shape[0] == len(ev) == ns[0]
    np.testing.assert_array_equal(rows[0], rrows)


class _PairLib:
    """grs_pair_spots with `per` rows an orientation, or with an error."""

    def __init__(self, per, error=0):
        self.per, self.error, self.caps = per, error, []

    def grs_pair_spots(self, h, pos, U, M, ns, ni, med, rp, rows, cap):
        self.caps.append(cap)
        rp[0] = 0
        if self.error:
            return self.error
        for m in range(M):
            rp[m + 1] = rp[m] + self.per
        return -1 if rp[M] > cap else 0


def _pair_engine(lib):
    from grainrecon_amd import Engine

    class Stub(Engine):
        def __init__(self):
            self._lib, self._h = lib, None

        def _chk(self, code):
            assert code == 0, code

    return Stub()


@pytest.mark.parametrize("per, M, calls", [(1024, 3, 1), (1025, 3, 2), (5, 2000, 1), (600, 2000, 2)])
def test_pair_spots_calls(per, M, calls):
    """One call where the first buffer (1024 rows an orientation, at most 2^20)
    holds the pairs, else a second one for exactly as many as there are."""
    lib = _PairLib(per)
    _, _, _, rows = _pair_engine(lib).pair_spots(np.zeros((M, 3)), np.zeros((M, 9)))
    assert len(lib.caps) == calls and lib.caps[0] == min(1024 * M, 1 << 20)
    assert calls == 1 or lib.caps[1] == per * M
    assert [r.shape for r in rows] == [(per, 23)] * M


@pytest.mark.parametrize("error", [-1, -3, -4])
def test_pair_spots_reports_an_error_at_once(error):
    lib = _PairLib(5, error)
    with pytest.raises(AssertionError, match=str(error)):
        _pair_engine(lib).pair_spots(np.zeros((3, 3)), np.zeros((3, 9)))
    assert len(lib.caps) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("nrot, M", [(37, 3), (6001, 131)])
def test_pair_spots_counts_beyond_the_capacity(engine, nrot, M):
    """A call whose rows do not fit still returns every row count, in one
    chunk of orientations and in two (2^26 / (6001 x 86) = 130 a chunk)."""
    from grainrecon_amd import _lib as L

    s = scenes.make_scene(seed=85, ngrains=1, spread_mm=0.02, nrot=nrot, det=32, pixel_mm=6.72e-3 * 32)
    engine.set_geometry(s.geo, s.hkl, s.rot)
    engine.set_distance_stack(np.zeros_like(s.proj))
    engine.set_frame_spots([np.array([[16.0, 16.0, 81.0]])] * nrot)
    pos, U = np.repeat(s.centers[:1], M, 0), np.repeat(np.reshape(s.U[0], (1, 9)), M, 0)
    _, _, _, rows = engine.pair_spots(pos, U)
    n = rows[0].shape[0]
    assert n > 0 and all(np.array_equal(r, rows[0]) for r in rows)
    out, rp = np.zeros((n, 23)), np.zeros(M + 1, np.int64)
    ns, ni, med = np.zeros(M, np.int32), np.zeros(M, np.int32), np.zeros(M, np.float32)
    p = lambda a: a.ctypes.data_as(ctypes.POINTER(np.ctypeslib.as_ctypes_type(a.dtype)))  # noqa: E731
    code = engine._lib.grs_pair_spots(engine._h, p(pos), p(U), M, p(ns), p(ni), p(med), p(rp), p(out), n)
    assert code == L.GRS_ERR_ARG and np.array_equal(rp, n * np.arange(M + 1))
    assert f"{M * n} pair rows do not fit" in engine._lib.grs_last_error(engine._h).decode()
