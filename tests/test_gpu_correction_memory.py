"""What the correction's pools take per voxel of the distance arena: for every eighth voxel a triangle record or
a row of a list (32 B), a barycenter (24 B), a row's source (4 B) and an eighth of a group's tag (2 B), 7.53 B, and
nothing more that grows with the arena; 8 B is what they took with boxed chunks instead of lists.  Two contexts that differ in the arena only; the free memory before and after."""
import ctypes

import numpy as np
import pytest

import gragles_3d_amd as G
import physics_cases as PC

pytestmark = pytest.mark.gpu


def _taken(case, arena):
    p, idf, bounds, exists, offs, ids = case
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    hip = ctypes.CDLL("libamdhip64.so")
    ctx = G.LevelSetContext(p, precision=G.FP32_BATCHED, arena_voxels=arena)
    ctx.set_boxes(bounds, exists)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    before = free.value
    ctx.set_physics(stored_energy=True, see=np.zeros(p.n_grains + 1))
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    ctx.close()
    return before - free.value


def test_pools_per_arena_voxel():
    print("correction pools: 27 grains, arenas of 3e7 and 2.3e8 voxels", flush=True)
    case = PC.voronoi_case(27, 10, 3, 5)
    small, large = _taken(case, 30_000_000), _taken(case, 230_000_000)
    per_voxel = (large - small) / 200e6
    assert 7.4 <= per_voxel <= 8.0, per_voxel  # (allocations are rounded up by up to a few MB each)
