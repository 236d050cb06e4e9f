"""The correction's nearest-element search against the oracle, FP64 bit for bit, where its layout can go
wrong: every box-size class (runs of 8, 4, 2 and 1 layers, sides that are no multiple of the run), grains
whose few barycenters fill partial groups, and a row pool too small for every slot's list (those slots
are searched without one).

Each case prints its name, seed and shape before touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
from oracle import oracle as O
import physics_cases as PC
from parity import compare_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_grains,ppg,border,seed,steps,tight", [
    (20, 21, 4, 3, 3, False),    # sides 33..48, ragged
    (8, 34, 5, 2, 2, False),     # sides above 48 and above 64
    (400, 7, 3, 6, 3, False),    # small grains: one group per element
    (1500, 6, 3, 4, 2, True),    # rows for fewer slots than there are
])
def test_search_equals_oracle(n_grains, ppg, border, seed, steps, tight):
    print("correction search: n=%d ppg=%d border=%d seed=%d steps=%d tight=%s" % (n_grains, ppg, border, seed, steps,
                                                                                  tight), flush=True)
    case = PC.voronoi_case(n_grains, ppg, border, seed)
    p, idf, bounds, exists, offs, ids = case
    side = np.max(bounds[1:, 3:] - bounds[1:, :3], axis=1).astype(np.int64)
    ctx = G.LevelSetContext(p, precision=G.FP64_PLAIN, arena_voxels=int(1.3 * np.sum(side ** 3)) if tight else 0)
    ctx.set_boxes(bounds, exists)
    ctx.init_distance(idf)
    ctx.set_neighbour_lists(offs, ids)
    orc = PC.oracle_sim(O, case)
    quat = PC.low_angle_orientations(n_grains, 11)
    see = G.lognormal_energies(n_grains, 3, median=0.1, sigma=1.0)
    phys = dict(mobility_model=True, unique_energies=False, stored_energy=True, quat=quat, see=see)
    ctx.set_physics(triple_line_drag=1e6, **phys)
    orc.set_physics(tl_drag=1e6, **phys)
    for s in range(steps):
        ctx.timestep(1)
        orc.timestep(1)
        compare_all(ctx, orc, "step %d" % s)
    ctx.close()
    orc.close()
