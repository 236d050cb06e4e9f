"""How full the pool of the correction's barycenter lists is (gg_get_correction_lists): refused before the
correction is on, 0 before the first hull, then what the grains' lists take, with room for all of them in an
arena of the default size.  In an arena too small for them some voxels are searched without a list: the same
results, FP64 as the oracle's bit for bit, FP32 as with lists bit for bit.  Each case prints its name before touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
from oracle import oracle as O
import physics_cases as PC
from parity import compare_all

pytestmark = pytest.mark.gpu


def _context(n_grains, ppg, border, seed, tight=0.0, precision=G.FP64_PLAIN):
    case = PC.voronoi_case(n_grains, ppg, border, seed)
    p, idf, bounds, exists, offs, ids = case
    side = np.max(bounds[1:, 3:] - bounds[1:, :3], axis=1).astype(np.int64)
    ctx = G.LevelSetContext(p, precision=precision, arena_voxels=int(tight * np.sum(side ** 3)))
    ctx.set_boxes(bounds, exists)
    ctx.init_distance(idf)
    ctx.set_neighbour_lists(offs, ids)
    return ctx, case


@pytest.mark.parametrize("n_grains,ppg,border,seed", [(8, 34, 5, 2), (64, 10, 3, 1), (1500, 6, 3, 4)])
def test_lists_of_default_arenas_have_room(n_grains, ppg, border, seed):
    print("correction lists: n=%d ppg=%d border=%d seed=%d" % (n_grains, ppg, border, seed), flush=True)
    ctx, _ = _context(n_grains, ppg, border, seed)
    with pytest.raises(G.GGError):
        ctx.correction_lists()
    ctx.set_physics(stored_energy=True, see=G.lognormal_energies(n_grains, 3))
    assert ctx.correction_lists()[0] == 0
    for _ in range(3):
        ctx.timestep(1)
        asked, room = ctx.correction_lists()
        assert n_grains <= asked <= room  # every grain borders something
    ctx.close()


def test_search_without_lists_equals_oracle():
    print("correction lists: n=1500 ppg=6 border=3 seed=4, an arena of 1.3 times the boxes", flush=True)
    ctx, case = _context(1500, 6, 3, 4, tight=1.3)
    orc = PC.oracle_sim(O, case)
    phys = dict(mobility_model=True, unique_energies=False, stored_energy=True, quat=PC.low_angle_orientations(1500, 11),
                see=G.lognormal_energies(1500, 3, median=0.1, sigma=1.0))
    ctx.set_physics(triple_line_drag=1e6, **phys)
    orc.set_physics(tl_drag=1e6, **phys)
    for s in range(3):
        ctx.timestep(1)
        orc.timestep(1)
        asked, room = ctx.correction_lists()
        assert asked > room, "every list found room"
        compare_all(ctx, orc, "step %d" % s)
    ctx.close()
    orc.close()


def test_search_without_lists_equals_search_with_them_fp32():
    print("correction lists: FP32, n=1500 ppg=6 border=3 seed=4, arenas of 1.3 and 2 times the boxes", flush=True)
    out = []
    for tight in (1.3, 0.0):
        ctx, _ = _context(1500, 6, 3, 4, tight=tight, precision=G.FP32_BATCHED)
        ctx.set_physics(mobility_model=True, unique_energies=False, quat=PC.low_angle_orientations(1500, 11))
        ctx.timestep(1)
        asked, room = ctx.correction_lists()
        assert (asked > room) == (tight > 0)
        ctx.timestep(4, use_graph=True)
        state = ctx.stats()[0]
        out.append((state, [ctx.phi(g, 1) for g in np.nonzero(state == G.ALIVE)[0]]))
        ctx.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for (b0, v0), (b1, v1) in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(b0, b1)
        np.testing.assert_array_equal(v0, v1)
