"""How full the pool of the correction's barycenter lists is (gg_get_correction_lists): refused before the
correction is on, 0 before the first hull, then what the grains' lists take, with room for all of them in an
arena of the default size.  Each case prints its name before touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
import physics_cases as PC

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
