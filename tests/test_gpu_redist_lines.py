"""Redistancing with whole lines in registers at the box sides where the unrolled length changes (33 to 48,
a step every 4), FP64, against the oracle bit for bit.  Two grains: a ball in its matrix, and a random field
(a sign change at about every second point of every line).  The volumes are not what is tested: 1e-9, for
the random field's signed terms cancel by up to a factor of 1e3.  Each case prints its name before touching the GPU.
"""
import pytest

from oracle import oracle as O
import physics_cases as PC
from parity import STAGE_SEQUENCE, compare_all, run_stage
from test_gpu_hull_edges import _random_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("random", [False, True])
@pytest.mark.parametrize("side", [33, 36, 37, 40, 41, 44, 45, 48])
def test_redistancing_at_line_lengths(side, random):
    print("redistancing lines: side %d, %s" % (side, "random field" if random else "ball"), flush=True)
    case = _random_pair(side - 5) if random else PC.sphere_in_matrix(side - 5)
    assert case[2][2][3] - case[2][2][0] == side
    ctx = PC.gpu_context(case)
    orc = PC.oracle_sim(O, case)
    for k in range(2):
        for name in STAGE_SEQUENCE:
            run_stage(ctx, name)
            run_stage(orc, name)
        compare_all(ctx, orc, "side %d step %d" % (side, k), rtol_stats=1e-9)
    ctx.close()
    orc.close()
