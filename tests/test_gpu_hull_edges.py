"""The hull against the oracle where its layout can go wrong: box sides at which a row of cells fills a
64-bit word, spills into a second part or ends a size class, and a field whose cells are nearly all cut
(every queue fills up).  Two grains, FP64, without and with topology.

Volume and area are compensated sums in another order than the oracle's: 1e-11 relative for the ball;
1e-9 for the random field, whose signed volume terms (about 1e6 of them, each rounded to 1e-16) cancel by
up to a factor of 1e3.

Each case prints its name and shape before touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
from oracle import oracle as O
import physics_cases as PC
from parity import compare_all
from test_gpu_topology import _compare

pytestmark = pytest.mark.gpu


def _random_pair(rds):
    p, idf, bounds, exists, offs, ids = PC.sphere_in_matrix(rds)
    inside = idf > 0
    idf = idf.copy()
    idf[inside] = np.random.default_rng(rds).integers(1, 3, size=int(inside.sum()))
    bounds[1] = bounds[2]
    return p, idf, bounds, exists, offs, ids


@pytest.mark.parametrize("topology", [False, True])
@pytest.mark.parametrize("side,random", [(48, False), (49, True), (63, False), (64, False), (65, True), (66, False),
                                         (96, False)])
def test_hull_at_word_and_class_edges(side, random, topology):
    print("hull edges: side %d, %s field, topology %s" % (side, "random" if random else "ball", topology), flush=True)
    case = _random_pair(side - 5) if random else PC.sphere_in_matrix(side - 5)
    p, idf, bounds, exists, offs, ids = case
    assert bounds[2][3] - bounds[2][0] == side
    ctx = PC.gpu_context(case)
    orc = PC.oracle_sim(O, case)
    ctx.enable_hull_topology(topology)
    ctx.timestep(1)
    orc.timestep(1)
    compare_all(ctx, orc, "side %d" % side, rtol_stats=1e-9 if random else 1e-11)
    if topology:
        assert _compare(ctx, orc, "side %d" % side) == 2
    ctx.close()
    orc.close()
