"""The FP32 redistancing at the box sides where a line's unrolled length changes (every 4 up to 48) against the
oracle's box function, bit for bit: on a field of +-h with h a power of two every value on the way is a small
multiple of h / 2 (the step across a sign change is h / 2), so nothing is rounded.  A ball in its matrix, and a
random field (a sign change at about every second point of every line).  Each case prints its name before
touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
from oracle import oracle as O
import physics_cases as PC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("random", [False, True])
@pytest.mark.parametrize("side", [17, 20, 21, 24, 25, 28, 29, 32, 33, 36, 37, 40, 41, 44, 45, 48])
def test_fp32_redistancing_at_line_lengths(side, random):
    print("FP32 redistancing lines: side %d, %s" % (side, "random field" if random else "ball"), flush=True)
    case = PC.sphere_in_matrix(side - 4, radius=(side - 11) / 2.0)  # the first step shrinks the outer box by one
    p = case[0]
    p.h, p.delta = 1.0 / 32, 3.0 / 32
    ctx = PC.gpu_context(case, precision=G.FP32_BATCHED)
    for name in ("switch", "convolution", "switch", "update_lists", "comparison", "switch", "level_set"):
        getattr(ctx, name)()
    rng = np.random.default_rng(side)
    want = {}
    for g in (1, 2):
        b, v = ctx.phi(g, 0)
        v = np.where(rng.random(v.size) < 0.5, -p.h, p.h) if random else np.where(v < 0, -p.h, p.h)
        ctx.upload_phi(g, 0, v)
        n = b[3] - b[0]
        want[g] = O.redistance_box(b, v.reshape(n, n, n), ctx.bounds(g, 1), p.h, p.delta)
    assert max(w.shape[0] for w in want.values()) == side
    ctx.redistancing()
    for g in (1, 2):
        np.testing.assert_array_equal(ctx.phi(g, 1)[1].reshape(want[g].shape), want[g])
    ctx.close()
