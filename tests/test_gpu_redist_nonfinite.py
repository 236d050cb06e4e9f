"""Redistancing of fields with NaN and infinities in them: a NaN has no sign (0), so a step past one adds
nothing, and no result is NaN.  Every form of the sweeps (two layers per wavefront, one layer, lines in LDS),
both precisions, against the oracle's box function on the same input, bit for bit: FP64 as it always is; FP32
on a field of +-h with h a power of two, where every value on the way is a small multiple of h / 2 (the step
across a sign change is h / 2), so nothing is rounded.

Each case prints its name before touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
from oracle import oracle as O
import physics_cases as PC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,precision", [(24, G.FP64_PLAIN), (31, G.FP64_PLAIN), (40, G.FP64_PLAIN),
                                            (48, G.FP64_PLAIN), (60, G.FP64_PLAIN), (21, G.FP32_BATCHED),
                                            (37, G.FP32_BATCHED), (69, G.FP32_BATCHED)])
def test_redistancing_of_nonfinite_input(side, precision):
    print("redistancing of non-finite input: side %d, precision %d" % (side, precision), flush=True)
    case = PC.sphere_in_matrix(side - 5)
    p = case[0]
    ctx = PC.gpu_context(case, precision=precision)
    for name in ("switch", "convolution", "switch", "update_lists", "comparison", "switch", "level_set"):
        getattr(ctx, name)()
    rng = np.random.default_rng(side)
    want = {}
    for g in (1, 2):
        b, v = ctx.phi(g, 0)
        v = v.copy() if precision == G.FP64_PLAIN else np.where(v < 0, -p.h, p.h)
        at = rng.choice(v.size, size=v.size // 20, replace=False)
        v[at] = rng.choice([np.nan, np.nan, np.inf, -np.inf], size=at.size)
        ctx.upload_phi(g, 0, v)
        n = b[3] - b[0]
        want[g] = O.redistance_box(b, v.reshape(n, n, n), ctx.bounds(g, 1), p.h, p.delta)
    ctx.redistancing()
    for g in (1, 2):
        assert not np.isnan(want[g]).any()
        np.testing.assert_array_equal(ctx.phi(g, 1)[1].reshape(want[g].shape), want[g])
    ctx.close()
