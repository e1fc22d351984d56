"""Small synthetic lab-DCT scenes for the tests.

Spot masks are rendered from the forward_comp geometry through the C oracle
(one pixel per selected event of every voxel of every grain), optionally
dilated, and turned into a bwdist-style Euclidean distance stack with scipy.
Sizes are chosen so the oracle finishes in seconds.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
from scipy import ndimage

import oracle
from grainrecon_amd.geometry import cubic_hkl, labdct_geometry


def random_quats(rng, n):
    """Haar-uniform unit quaternions (Shoemake 1992) with q0 >= 0."""
    u1, u2, u3 = rng.random((3, n))
    q = np.stack([np.sqrt(1 - u1) * np.sin(2 * np.pi * u2), np.sqrt(1 - u1) * np.cos(2 * np.pi * u2),
                  np.sqrt(u1) * np.sin(2 * np.pi * u3), np.sqrt(u1) * np.cos(2 * np.pi * u3)], axis=1)
    q[q[:, 0] < 0] *= -1
    return q


def U_from_qvec(q1, q2, q3):
    """U exactly as the engine builds it: q0 recomputed from the vector part
    (ForwardCalc_OR_space_comp.m:27-49), same operation order."""
    ss = (q1 * q1 + q2 * q2) + q3 * q3
    q0 = math.sqrt(1.0 - ss)
    return np.array([
        [2.0 * (q0 * q0 + q1 * q1) - 1.0, 2.0 * (q1 * q2 - q0 * q3), 2.0 * (q1 * q3 + q0 * q2)],
        [2.0 * (q1 * q2 + q0 * q3), 2.0 * (q0 * q0 + q2 * q2) - 1.0, 2.0 * (q2 * q3 - q0 * q1)],
        [2.0 * (q1 * q3 - q0 * q2), 2.0 * (q2 * q3 + q0 * q1), 2.0 * (q0 * q0 + q3 * q3) - 1.0],
    ])


def free_device_memory(engine):
    """Bytes free on the device, from the HIP runtime the engine's library is linked to."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert engine._lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


class Scene:
    pass


def make_scene(seed=0, det=256, pixel_mm=6.72e-3 * 4, nrot=37, families=6, lattice="I", a=2.8665, ngrains=3,
               grain_vox=3, vox_mm=0.005, spread_mm=0.06, dilate=1, tilts=(0.0, 0.0, 0.0), dety00=0.0, detz00=0.0,
               beamstop=((0.0, -1.0), (0.0, -1.0))):
    rng = np.random.default_rng(seed)
    s = Scene()
    s.geo = labdct_geometry(a=a, lattice=lattice, det_pixels=det, pixel_mm=pixel_mm, tilts=tilts, dety00=dety00,
                            detz00=detz00, beamstop=beamstop)
    s.hkl = cubic_hkl(lattice, families)
    s.rot = np.linspace(0.0, 360.0, nrot)
    s.q = random_quats(rng, ngrains)
    s.U = [U_from_qvec(*s.q[g, 1:]) for g in range(ngrains)]
    s.centers = rng.uniform(-spread_mm, spread_mm, (ngrains, 3))
    offs = (np.arange(grain_vox) - (grain_vox - 1) / 2) * vox_mm
    grid = np.stack(np.meshgrid(offs, offs, offs, indexing="ij"), -1).reshape(-1, 3)
    s.voxels = [c + grid for c in s.centers]
    mask = np.zeros((det, det, nrot), dtype=bool)
    zero = oracle.Stack(np.zeros((det, det, nrot), np.float32))
    for g in range(ngrains):
        for p in s.voxels[g]:
            _, _, _, ev = oracle.forward_comp(s.geo, zero, s.U[g], p, s.rot, s.hkl, events=True)
            for om, _h, dy, dz, *_ in ev:
                mask[int(dz) - 1, int(dy) - 1, int(om)] = True
    if dilate:
        st = ndimage.generate_binary_structure(2, 1)
        for i in range(nrot):
            mask[:, :, i] = ndimage.binary_dilation(mask[:, :, i], st, iterations=dilate)
    s.mask = mask
    dist = np.zeros(mask.shape, np.float32)
    for i in range(nrot):
        if mask[:, :, i].any():
            dist[:, :, i] = ndimage.distance_transform_edt(~mask[:, :, i]).astype(np.float32)
        else:
            dist[:, :, i] = np.float32(det)  # no spot on this projection
    s.proj = dist
    s.stack = oracle.Stack(dist)
    return s
