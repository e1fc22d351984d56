"""Orientation fit (fit_OR_constrain_with_local_comp_cuda.m:116-126): the
batched device fit against the sequential oracle fit, step for step."""
import numpy as np
import pytest

import oracle
import scenes
from oracle.fit_or import fit_or_local, objective


@pytest.fixture(scope="module")
def scene():
    return scenes.make_scene(seed=33, ngrains=3, spread_mm=0.05, nrot=37)


def _starts(s, rng, k):
    pos, x0 = [], []
    for i in range(k):
        g = i % 3
        pos.append(s.voxels[g][int(rng.integers(0, 27))])
        x0.append(s.q[g, 1:] + rng.uniform(-0.006, 0.006, 3))
    return np.array(pos), np.array(x0)


def test_oracle_fit_improves_completeness(scene):
    s = scene
    rng = np.random.default_rng(1)
    pos, x0 = _starts(s, rng, 1)
    f0 = objective(s.geo, s.stack, pos[0], x0[0], s.rot, s.hkl)
    x, fv, nf, it = fit_or_local(s.geo, s.stack, pos[0], x0[0], s.rot, s.hkl)
    assert fv <= f0 and nf <= 2000 + 3
    assert np.all(np.abs(x - x0[0]) <= 0.02)
    assert fv == objective(s.geo, s.stack, pos[0], x, s.rot, s.hkl)


def test_oracle_fit_respects_budget(scene):
    s = scene
    pos, x0 = _starts(s, np.random.default_rng(2), 1)
    _, _, nf, it = fit_or_local(s.geo, s.stack, pos[0], x0[0], s.rot, s.hkl, max_fun_evals=12)
    assert nf <= 12 + 3


@pytest.mark.gpu
def test_batched_fit_equals_sequential_oracle(engine, scene):
    s = scene
    engine.set_geometry(s.geo, s.hkl, s.rot)
    engine.set_distance_stack(s.proj)
    rng = np.random.default_rng(3)
    pos, x0 = _starts(s, rng, 6)
    x0[5] = [0.9, 0.5, 0.3]          # |q_vec| > 1 everywhere near it: NaN objective
    x, fv, nf, it = engine.fit_or_local(pos, x0)
    for m in range(pos.shape[0]):
        rx, rf, rnf, rit = fit_or_local(s.geo, s.stack, pos[m], x0[m], s.rot, s.hkl)
        np.testing.assert_array_equal(x[m], rx)
        assert (fv[m] == rf) or (np.isnan(fv[m]) and np.isnan(rf))
        assert nf[m] == rnf and it[m] == rit
    assert np.sum(fv[:5] < 0.5) >= 3 and np.isnan(fv[5]) and nf[5] >= 2000


@pytest.mark.gpu
@pytest.mark.parametrize("H", [1, 3, 85, 86])
def test_fits_with_uneven_reflection_shares(engine, scene, H):
    """Reflection counts that split unevenly over a team's waves (some left
    without any), with the hits read from the keys and from the bit mask
    (which a counts-only call builds): each fit equals the sequential one."""
    s = scene
    hkl = s.hkl[:H]
    engine.set_geometry(s.geo, hkl, s.rot)
    engine.set_distance_stack(s.proj)
    pos, x0 = _starts(s, np.random.default_rng(H), 3)
    ref = [fit_or_local(s.geo, s.stack, pos[m], x0[m], s.rot, hkl, max_fun_evals=60) for m in range(3)]
    for _ in range(2):
        x, fv, nf, it = engine.fit_or_local(pos, x0, max_fun_evals=60)
        for m, (rx, rf, rnf, rit) in enumerate(ref):
            np.testing.assert_array_equal(x[m], rx)
            assert (fv[m] == rf or (np.isnan(fv[m]) and np.isnan(rf))) and nf[m] == rnf and it[m] == rit
        engine.compete_csr(pos[:1], [0, 1], s.q[:1], 2, 0.004)


@pytest.mark.gpu
def test_fit_longer_than_one_launch(engine, scene):
    """A fit whose every value is NaN shrinks at each iteration: 4 + 5 k
    evaluations after k iterations, so 20,000 end it at 20,004 in iteration
    4,001, more requests than one launch serves."""
    s = scene
    engine.set_geometry(s.geo, s.hkl, s.rot)
    engine.set_distance_stack(s.proj)
    pos, x0 = _starts(s, np.random.default_rng(5), 2)
    x0[1] = [0.9, 0.5, 0.3]
    x, fv, nf, it = engine.fit_or_local(pos, x0, max_fun_evals=20000, max_iter=1000000)
    assert np.isnan(fv[1]) and nf[1] == 20004 and it[1] == 4001
    rx, rf, rnf, rit = fit_or_local(s.geo, s.stack, pos[0], x0[0], s.rot, s.hkl, max_fun_evals=20000, max_iter=1000000)
    np.testing.assert_array_equal(x[0], rx)
    assert fv[0] == rf and nf[0] == rnf and it[0] == rit


@pytest.mark.gpu
def test_large_batches_bound_their_tables():
    """8,000 fits at 1,441 angles run in launches whose beam tables take at
    most 512 MB (1.1 GB in one launch), with the results of small calls around
    the launches' ends."""
    from grainrecon_amd import Engine

    s = scenes.make_scene(seed=61, ngrains=2, spread_mm=0.03, nrot=1441, det=64, pixel_mm=6.72e-3 * 16)
    rng = np.random.default_rng(7)
    pos = s.centers[rng.integers(0, 2, 8000)] + rng.uniform(-0.01, 0.01, (8000, 3))
    x0 = s.q[rng.integers(0, 2, 8000), 1:] + rng.normal(scale=2e-3, size=(8000, 3))
    e = Engine(0)
    try:
        e.set_geometry(s.geo, s.hkl[:8], s.rot)
        e.set_distance_stack(s.proj)
        e.fit_or_local(pos[:5], x0[:5], max_fun_evals=10)
        free = scenes.free_device_memory(e)
        got = e.fit_or_local(pos, x0, max_fun_evals=10)
        assert free - scenes.free_device_memory(e) < 700 << 20
        most = (512 << 20) // (96 * 1441)
        for part in (slice(0, 5), slice(most - 3, most + 3), slice(2 * most - 3, 2 * most + 3), slice(7995, 8000)):
            for a, b in zip(got, e.fit_or_local(pos[part], x0[part], max_fun_evals=10)):
                np.testing.assert_array_equal(a[part], b)
    finally:
        e.close()
