"""The correction where every size class is a branch of its own (boxes of 50 MB and more: 1.6e7 voxels here), on a
case with boxes of all four size classes: the convolution and correction of the classes run beside each other and
beside the list build and the IDLocal resize.  FP64, eager and captured steps, against the oracle bit for bit; FP32
against the same run on one stream (as stage timing has it), bit for bit.  And what the FP32 correction does
to boxes above 32, from a second context without it: every band voxel moves by the weights of one of the elements
that border its id.

Each case prints its name before touching the GPU.
"""
import numpy as np
import pytest

import gragles_3d_amd as G
from oracle import oracle as O
import physics_cases as PC
from parity import compare_all

pytestmark = pytest.mark.gpu

N, PPG, BORDER, SEED = 216, 26, 3, 1


@pytest.fixture(scope="module")
def case():
    c = PC.voronoi_case(N, PPG, BORDER, SEED)
    side = np.max(c[2][1:, 3:] - c[2][1:, :3], axis=1)
    assert all(((side > a) & (side <= b)).any() for a, b in ((0, 32), (32, 48), (48, 64), (64, 96))), side
    assert np.sum(side.astype(np.int64) ** 3) * 4 > 50_000_000  # FP32 too
    return c


def _physics():
    return dict(mobility_model=True, unique_energies=False, stored_energy=True,
                quat=PC.low_angle_orientations(N, 11), see=G.lognormal_energies(N, 3, median=0.1, sigma=1.0))


def _context(case, precision, correction=True):
    p, idf, bounds, exists, offs, ids = case
    ctx = G.LevelSetContext(p, precision=precision)
    ctx.set_boxes(bounds, exists)
    ctx.init_distance(idf)
    ctx.set_neighbour_lists(offs, ids)
    if correction:
        ctx.set_physics(triple_line_drag=1e6, **_physics())
    return ctx


def test_branches_fp64_equal_oracle(case):
    print("correction branches: FP64, n=%d ppg=%d border=%d seed=%d" % (N, PPG, BORDER, SEED), flush=True)
    ctx = _context(case, G.FP64_PLAIN)
    orc = PC.oracle_sim(O, case)
    orc.set_physics(tl_drag=1e6, **_physics())
    for step in range(2):
        ctx.timestep(1)
        orc.timestep(1)
        compare_all(ctx, orc, "eager step %d" % step)
    for replay in range(2):
        ctx.timestep(2, use_graph=True)
        ctx.synchronize()
        orc.timestep(2)
        compare_all(ctx, orc, "replay %d" % replay)
    ctx.close()
    orc.close()


def test_branches_follow_the_boxes_set(case):
    """One context: first few of the grains (no branches), captured steps, then all of them (branches)."""
    print("correction branches: boxes set twice, n=%d ppg=%d" % (N, PPG), flush=True)
    p, idf, bounds, exists, offs, ids = case
    ctx = G.LevelSetContext(p, precision=G.FP64_PLAIN, arena_voxels=2 * int(np.sum(
        np.max(bounds[1:, 3:] - bounds[1:, :3], axis=1).astype(np.int64) ** 3)))
    few = exists.copy()
    few[40:] = 0
    for some in (few, exists):
        o, i = G.initial_neighbour_lists(p, bounds, some)
        ctx.set_boxes(bounds, some)
        ctx.set_physics(triple_line_drag=1e6, **_physics())
        orc = PC.oracle_sim(O, (p, idf, bounds, some, o, i))
        orc.set_physics(tl_drag=1e6, **_physics())
        ctx.init_distance(idf)
        ctx.set_neighbour_lists(o, i)
        ctx.timestep(3, use_graph=True)
        orc.timestep(3)
        compare_all(ctx, orc, "%d grains" % int(some.sum()))
        orc.close()
    ctx.close()


@pytest.mark.parametrize("graph", [False, True])
def test_branches_fp32_equal_one_stream(case, graph):
    print("correction branches: FP32, %s, n=%d ppg=%d" % ("captured" if graph else "eager", N, PPG), flush=True)
    out = []
    for one_stream in (False, True):
        ctx = _context(case, G.FP32_BATCHED)
        ctx.enable_stage_timing(one_stream)
        ctx.timestep(6, use_graph=graph)
        state = ctx.stats()[0]
        out.append((state, [ctx.phi(g, 1) for g in np.nonzero(state == G.ALIVE)[0]]))
        ctx.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for (b0, v0), (b1, v1) in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(b0, b1)
        np.testing.assert_array_equal(v0, v1)


def test_fp32_correction_uses_weights_of_bordering_elements(case):
    print("correction weights: FP32, n=%d ppg=%d, boxes above 32" % (N, PPG), flush=True)
    p, idf, bounds, exists, offs, ids = case
    a = _context(case, G.FP32_BATCHED, correction=False)
    a.set_physics(mobility_model=True, unique_energies=False, triple_line_drag=1e6, quat=_physics()["quat"])
    b = _context(case, G.FP32_BATCHED, correction=False)
    for ctx in (a, b):
        ctx.timestep(1)  # the first step has no correction
        ctx.switch()
        ctx.convolution()
    checked = moved = 0
    for g in range(1, N + 1):
        box, before = a.phi(g, 0)
        if box[3] - box[0] <= 32:
            continue
        np.testing.assert_array_equal(before, b.phi(g, 0)[1])
        got, plain = a.phi(g, 1)[1], b.phi(g, 1)[1]
        old = a.idlocal(g)[1]
        idl = np.zeros(before.size, dtype=np.int64)  # the old content at the same linear index
        idl[:min(old.size, idl.size)] = old[:idl.size]
        band = np.abs(before) < p.delta
        np.testing.assert_array_equal(got[~band], plain[~band])
        el = a.correction_elements(g)
        for i in np.unique(idl[band]):
            at = band & (idl == i)
            w = {(m, e) for nb, m, e in zip(el["nb"], el["mobility"], el["energy"]) if int(i) in nb} or {(1.0, 1.0)}
            hit = np.zeros(int(at.sum()), dtype=bool)
            for m, e in w:
                hit |= got[at] == (before[at] + (plain[at] - before[at]) * m * e).astype(np.float32)
            assert hit.all(), "grain %d id %d: %d of %d" % (g, i, (~hit).sum(), hit.size)
            checked += hit.size
        moved += int((got[band] != plain[band]).sum())
    assert checked > 100000 and moved > checked // 4, (checked, moved)
    a.close()
    b.close()
