"""Interfacial elements where the merge of junctions has the most to do: a ball in 40 or 55 grains whose
seeds lie on a sphere around it, so that its hull has about 75 or 95 quadruple junctions (more than the
64 that are tested at a time), many within 2 voxels of each other.  Elements and the step's fields against
the oracle; the positions are sums in another order (1e-9, as in the other element tests).

Each case prints its name and shape before touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
from oracle import oracle as O
import physics_cases as PC
from parity import compare_all
from test_gpu_correction import _compare_elements

pytestmark = pytest.mark.gpu


def _ball_in_grains(k, rds=36, border=3, radius=10.0):
    p, idf, _, _, _, _ = PC.sphere_in_matrix(rds, border, radius)
    i = np.arange(k) + 0.5
    polar, azimuth = np.arccos(1 - 2 * i / k), np.pi * (1 + 5 ** 0.5) * i
    seeds = np.stack([np.cos(azimuth) * np.sin(polar), np.sin(azimuth) * np.sin(polar), np.cos(polar)], axis=1)
    seeds += np.random.default_rng(k).normal(0, 0.08, seeds.shape)
    seeds /= np.linalg.norm(seeds, axis=1, keepdims=True)
    c = (rds + 2 * border - 2) / 2.0
    zz, yy, xx = np.nonzero(idf == 2)
    pts = np.stack([xx - c, yy - c, zz - c], axis=1)
    pts /= np.maximum(np.linalg.norm(pts, axis=1, keepdims=True), 1e-9)
    idf = idf.copy()
    idf[zz, yy, xx] = 2 + np.argmax(pts @ seeds.T, axis=1)
    n = k + 1
    p.n_grains = n
    ngp = p.ngridpoints
    bounds = np.zeros((n + 1, 6), dtype=np.int32)
    exists = np.zeros(n + 1, dtype=np.uint8)
    for g in range(1, n + 1):
        z, y, x = np.nonzero(idf == g)
        lo = np.array([x.min(), y.min(), z.min()]) - border
        hi = np.array([x.max(), y.max(), z.max()]) + 1 + border
        side = int(min((hi - lo).max(), ngp))
        lo = np.clip(lo, 0, ngp - side)
        bounds[g] = [*lo, *(lo + side)]
        exists[g] = 1
    offs, ids = G.initial_neighbour_lists(p, bounds, exists)
    return p, idf, bounds, exists, offs, ids


@pytest.mark.parametrize("k", [40, 55])
def test_many_junctions_merge_as_in_the_oracle(k):
    print("junction merge: a ball in %d grains" % k, flush=True)
    case = _ball_in_grains(k)
    ctx = PC.gpu_context(case)
    orc = PC.oracle_sim(O, case)
    quat = PC.low_angle_orientations(k + 1, 11)
    phys = dict(mobility_model=True, unique_energies=False, stored_energy=False, quat=quat, see=None)
    ctx.set_physics(triple_line_drag=1e6, **phys)
    orc.set_physics(tl_drag=1e6, **phys)
    for s in range(2):
        ctx.timestep(1)
        orc.timestep(1)
        compare_all(ctx, orc, "step %d" % s)
        assert _compare_elements(ctx, orc, "step %d" % s) > 0
    assert sum(1 for e in orc.correction_elements(1) if e[0] == 3) > 0
    ctx.close()
    orc.close()
