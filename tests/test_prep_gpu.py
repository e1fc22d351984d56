"""GPU input preparation: spot rendering and the exact distance transform."""
import ctypes

import numpy as np
import pytest
from scipy import ndimage

import oracle
import scenes

pytestmark = pytest.mark.gpu


def test_render_matches_oracle_rendering(engine):
    s = scenes.make_scene(seed=71, ngrains=3, dilate=0)
    engine.set_geometry(s.geo, s.hkl, s.rot)
    pos = np.vstack(s.voxels)
    grain = np.repeat(np.arange(3), [len(v) for v in s.voxels])
    engine.render_spots(pos, grain, np.stack(s.U))
    got = engine.get_mask(s.mask.shape).astype(bool)
    assert got.sum() > 100
    assert np.array_equal(got, s.mask)


def test_edt_matches_scipy_bitwise(engine):
    rng = np.random.default_rng(3)
    s = scenes.make_scene(seed=72, ngrains=1, det=128, pixel_mm=6.72e-3 * 8, nrot=7)
    mask = rng.random((128, 96, 7)) < 0.01
    mask[:, :, 3] = False  # an empty projection
    mask[5, 7, 5] = True
    engine.set_geometry(s.geo, s.hkl, s.rot)
    engine.set_binary_stack(mask)
    engine.distance_from_mask()
    d = engine.get_distance_stack(mask.shape)
    for i in range(mask.shape[2]):
        if mask[:, :, i].any():
            ref = ndimage.distance_transform_edt(~mask[:, :, i]).astype(np.float32)
            assert np.array_equal(d[:, :, i].view(np.uint32), ref.view(np.uint32)), i
        else:
            assert np.isinf(d[:, :, i]).all()


@pytest.mark.parametrize("nz, ny", [(1, 1), (63, 16), (64, 17), (65, 33), (129, 250), (20, 1203), (70, 1204), (33, 2409),
                                    (17, 4817), (4096, 18), (4097, 18)])
def test_edt_at_tile_edges(engine, nz, ny):
    """Tile widths, partial tiles, row counts around the steps and the sides
    where another kernel takes over; few spots (long searches), many, none."""
    rng = np.random.default_rng(nz * 10007 + ny)
    mask = np.zeros((nz, ny, 4), bool)
    mask[rng.integers(nz), rng.integers(ny), 0] = True
    mask[:, :, 1] = rng.random((nz, ny)) < 3.0 / (nz * ny)
    mask[:, :, 2] = rng.random((nz, ny)) < 0.02
    mask[0, 0, 2] = True
    engine.set_binary_stack(mask)
    engine.distance_from_mask()
    d = engine.get_distance_stack(mask.shape)
    for i in range(4):
        if mask[:, :, i].any():
            ref = ndimage.distance_transform_edt(~mask[:, :, i]).astype(np.float32)
        else:
            ref = np.full((nz, ny), np.inf, np.float32)
        assert np.array_equal(d[:, :, i].view(np.uint32), ref.view(np.uint32)), i


@pytest.mark.parametrize("extra", [0, 1, 5])
def test_large_transfers_keep_every_byte(engine, extra):
    """Stacks and volumes above the size that goes through the staging
    threads, with a last chunk that is whole, nearly whole or short."""
    rng = np.random.default_rng(extra)
    nz, ny, nrot = 1024, 1024, 14 + extra
    d = rng.random((nrot, ny, nz + extra), dtype=np.float32).transpose(2, 1, 0)
    engine.set_distance_stack(d)
    assert np.array_equal(engine.get_distance_stack(d.shape), d)
    v = rng.random((256 + extra, 256, 160 + extra))
    engine.set_volume("Mask", v)
    assert np.array_equal(engine.get_volume("Mask"), v)
    m = rng.random((48 + extra, ny, nz)) < 0.5
    engine.set_binary_stack(m.transpose(2, 1, 0))
    assert np.array_equal(engine.get_mask((nz, ny, 48 + extra)), m.transpose(2, 1, 0))


def test_pinned_host_memory_is_copied_directly():
    """A stack in memory that the caller pinned goes to the device in one
    copy: no staging buffers (64 MB) and threads, which made it slower (15.4
    instead of 13.5 ms for 759 MB); one in pageable memory still has them."""
    from grainrecon_amd import Engine

    nz, ny, nrot = 1024, 1024, 16

    def address_space():
        return next(int(x.split()[1]) << 10 for x in open("/proc/self/status") if x.startswith("VmSize"))

    e = Engine(0)
    p = ctypes.c_void_p()
    assert e._lib.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(4 * nz * ny * nrot), 0) == 0
    try:
        pinned = np.frombuffer((ctypes.c_float * (nz * ny * nrot)).from_address(p.value), np.float32)
        rng = np.random.default_rng(9)
        pinned[:] = rng.random(pinned.size, dtype=np.float32)
        pageable = pinned + 1
        mask = np.zeros((nz, ny, nrot), bool)
        mask[3, 4] = True
        e.set_binary_stack(mask)  # the stack's buffer, and what the first copies allocate
        e.distance_from_mask()
        e.set_distance_stack(pinned[:nz * ny].reshape(1, ny, nz).transpose(2, 1, 0))
        shape = (nz, ny, nrot)
        for src, low, high in ((pinned, -(1 << 30), 32 << 20), (pageable, 60 << 20, 1 << 40)):
            used = address_space()
            e.set_distance_stack(src.reshape(shape[::-1]).transpose(2, 1, 0))
            assert low < address_space() - used < high
        assert np.array_equal(e.get_distance_stack(shape).ravel(order="F"), pageable)
        e.set_distance_stack(pinned.reshape(shape[::-1]).transpose(2, 1, 0))
        assert np.array_equal(e.get_distance_stack(shape).ravel(order="F"), pinned)
    finally:
        e.close()
        assert e._lib.hipHostFree(p) == 0


def test_rendered_scene_scores_one_at_truth(engine):
    s = scenes.make_scene(seed=73, ngrains=3, dilate=1)
    engine.set_geometry(s.geo, s.hkl, s.rot)
    pos = np.vstack(s.voxels)
    grain = np.repeat(np.arange(3), [len(v) for v in s.voxels])
    engine.render_spots(pos, grain, np.stack(s.U))
    engine.distance_from_mask()
    ns, ni, C, med = engine.forward_comp(s.centers[0], s.q)
    assert C[0] == 1.0 and med[0] == 0.0
    # the stack built on the GPU scores exactly as the oracle on the same stack
    stack = oracle.Stack(engine.get_distance_stack(s.mask.shape))
    ref = oracle.or_space_comp(s.geo, stack, s.centers[0], s.q, s.rot, s.hkl)
    assert np.array_equal(ns, ref[:, 0]) and np.array_equal(C.view(np.uint64), ref[:, 2].view(np.uint64))
