"""Timing cases of the per-grain level-set timestep.

A pass is one simulation segment as a user's program runs it on a context it
keeps: the boxes and the initial distance field of a microstructure go in
(gg_set_boxes, gg_init_distance), the neighbour lists are built on the device,
the timesteps run, and what the program reads afterwards comes back: grain
states, volumes, surface areas, box bounds, the grain count of every step, and
per case the distance fields, the faces and the id container.  A segment
starts from the same inputs each time, so a pass can be repeated.

prepare() makes the microstructure (host code of the library) and the context
with its options; run() is the pass.
"""
import math

import numpy as np

import gragles_3d_amd as G

# kind      voronoi: uniform-random seeds; bimodal: 10 % of the grains four times larger (power diagram)
# physics   none: isotropic; aniso: Read-Shockley energies and sigmoidal mobilities of a textured
#           orientation set; stored: isotropic boundaries with lognormal stored energies
# conv      default: FFT (FP64) or circulant (FP32); bf16: split-BF16 products (FP32 only)
# read      stats: states, volumes, areas, bounds and counts; container: also the id container; fields:
#           also every grain's distance field; topology: also the hull's faces (topology on) and the container
_BASE = {"kind": "voronoi", "border": 3, "physics": "none", "conv": "default", "graph": True, "read": "stats"}


def _case(name, **kw):
    return dict(_BASE, name=name, **kw)


def listed():
    return [
        # the smallest call: a smoke-sized domain in the default precision, stepped eagerly, fields read
        # back; latency and the number of launches count
        _case("fields_27_fp64", grains=27, ppg=12, fp32=False, steps=24, graph=False, read="fields"),
        # the same in the batched precision, odd box sides, captured steps
        _case("fields_30_fp32", grains=30, ppg=13, border=4, fp32=True, steps=24, read="fields"),
        # a small interactive run
        _case("small_216_fp32", grains=216, ppg=16, fp32=True, steps=60),
        # the plain reference workload: 512 grains, 16 points per grain, FP64
        _case("plain_512_fp64", grains=512, ppg=16, fp32=False, steps=50, read="container"),
        # few grains finely resolved: ragged boxes of side 45 to 80, the large size classes
        _case("fine_77_fp64", grains=77, ppg=31, border=5, fp32=False, steps=16, read="container"),
        # the headline workload in both precisions
        _case("headline_8000_fp32", grains=8000, ppg=20, fp32=True, steps=30),
        _case("headline_8000_fp64", grains=8000, ppg=20, fp32=False, steps=16),
        # bimodal grain sizes: box sides from 8 to 60 in one batch
        _case("uneven_20000_fp32", kind="bimodal", grains=20000, ppg=16, fp32=True, steps=16),
        # misorientation-dependent boundaries: the convolution correction, both precisions
        _case("aniso_4000_fp32", grains=4000, ppg=20, fp32=True, physics="aniso", steps=8, read="container"),
        _case("aniso_343_fp64", grains=343, ppg=17, fp32=False, physics="aniso", steps=20, read="container"),
        # stored-energy driven growth with the split-BF16 convolution
        _case("stored_20000_fp32", grains=20000, ppg=20, fp32=True, physics="stored", conv="bf16", steps=4),
        # an analysis run: hull topology every step, faces and the id container at the end
        _case("analysis_2000_fp32", grains=2000, ppg=18, fp32=True, steps=16, read="topology"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    case = dict(_BASE)
    case["kind"] = rng.choice(["voronoi", "voronoi", "voronoi", "bimodal"])
    case["fp32"] = rng.random() < 0.6
    case["physics"] = rng.choice(["none", "none", "aniso", "stored"])
    if case["kind"] == "bimodal":  # a large grain may touch more grains than a hull table holds
        case["physics"] = "none"
    case["border"] = rng.choice([3, 3, 4, 5])
    case["ppg"] = rng.randint(10, 16) if case["kind"] == "bimodal" else rng.randint(10, 30)
    lo = 300 if case["kind"] == "bimodal" else 20
    hi = 4000 if case["physics"] == "aniso" else 12000
    # voxel-updates of a pass stay well below those of the largest listed case; the correction and
    # FP64 cost more per voxel-update
    budget = (3.0e8 if case["physics"] != "none" else 1.5e9) * (1.0 if case["fp32"] else 0.5)
    case["grains"] = _log_int(rng, lo, hi)
    case["steps"] = rng.randint(4, 24)
    while voxels(case) * case["steps"] > budget:
        if case["steps"] > 4:
            case["steps"] = max(4, case["steps"] // 2)
        else:
            case["grains"] = max(lo, case["grains"] * 2 // 3)
            if case["grains"] == lo:
                break
    case["conv"] = "bf16" if case["fp32"] and rng.random() < 0.25 else "default"
    case["graph"] = rng.random() < 0.75
    case["read"] = "fields" if case["grains"] <= 64 else rng.choice(["stats", "container", "topology"])
    if case["kind"] == "bimodal" and case["read"] == "topology":
        case["read"] = "container"
    return case


def voxels(case):
    """Voxels of all boxes (their mean side follows the resolution and the border)."""
    return case["grains"] * ((1.09 if case["kind"] == "bimodal" else 1.28) * case["ppg"] + 2 * case["border"]) ** 3


def work(case):
    """Per step every voxel's distance and neighbour id are read once and written once and its convolution is an FFT
    there and back; the id field goes in once."""
    v = voxels(case)
    side = (v / case["grains"]) ** (1.0 / 3.0)
    esz = 4 if case["fp32"] else 8
    grid = G.derive_params(case["grains"], case["ppg"], case["border"]).ngridpoints ** 3
    return {"bytes": case["steps"] * v * (2 * esz + 8) + 4 * grid,
            "flops": case["steps"] * v * (2 * 2.5 * 3 * math.log2(side) + 30)}


def _microstructure(case, seed):
    p = G.derive_params(case["grains"], case["ppg"], case["border"])
    if case["kind"] == "bimodal":
        xyz, radius = G.bimodal_seeds(case["grains"], seed)
        idfield, bounds, exists = G.generate_power(p, xyz, radius)
    else:
        idfield, bounds, exists = G.generate_voronoi(p, seed)
    return p, idfield, bounds, exists


def _field_room(case):
    return int(2 * voxels(case))


def _padded(parts, room, fill, dtype):
    """The parts back to back in an array of a fixed length (how many values there are depends on the microstructure)."""
    out = np.full(room, fill, dtype=dtype)
    at = 0
    for v in parts:
        out[at:at + v.size] = v
        at += v.size
    return out


def prepare(case, seed):
    p, idfield, bounds, exists = _microstructure(case, seed)
    ctx = G.LevelSetContext(p, precision=G.FP32_BATCHED if case["fp32"] else G.FP64_PLAIN)
    ctx.set_boxes(bounds, exists)  # sizes the arenas
    if case["physics"] == "aniso":
        ctx.set_physics(mobility_model=True, unique_energies=False, triple_line_drag=1.0,
                        quat=G.textured_orientations(case["grains"], seed))
    elif case["physics"] == "stored":
        ctx.set_physics(stored_energy=True, triple_line_drag=1.0, see=G.lognormal_energies(case["grains"], seed))
    if case["conv"] == "bf16":
        ctx.set_convolution_form(G.CONV_SPLIT_BF16)
    if case["grains"] >= 2000:
        ctx.set_comparison_order(G.CMP_ORDER_SPACE, 1)  # what the autotuner picks at such sizes
    if case["read"] == "topology":
        ctx.enable_hull_topology()
    return {"ctx": ctx, "idfield": idfield, "bounds": bounds, "exists": exists, "steps": case["steps"],
            "graph": case["graph"], "read": case["read"], "dtype": np.float32 if case["fp32"] else np.float64,
            "field_room": _field_room(case), "face_room": 16 * case["grains"]}


def run(state):
    ctx = state["ctx"]
    ctx.set_boxes(state["bounds"], state["exists"])
    ctx.init_distance(state["idfield"])
    ctx.build_neighbour_lists()
    ctx.timestep(state["steps"], use_graph=state["graph"])
    grain, volume, area = ctx.stats()
    out = {"state": grain, "volume": volume, "area": area, "bounds": ctx.all_bounds(1),
           "counts": ctx.count_history()[-state["steps"]:]}
    if state["read"] == "fields":
        out["phi"] = _padded((ctx.phi(g, 1)[1] for g in np.nonzero(grain == G.ALIVE)[0]), state["field_room"], 0.0,
                             state["dtype"])
    elif state["read"] == "topology":
        a, b, face_area = ctx.faces()
        room = state["face_room"]
        out["faces"] = [_padded([a], room, -1, np.int32), _padded([b], room, -1, np.int32)]
        out["face_area"] = _padded([face_area], room, 0.0, np.float64)
    if state["read"] in ("container", "topology"):
        out["container"] = ctx.voxel_container()
    return out


# ---- the same segment in plain numpy, 64 bits (isotropic, small cases) ------------------------------

def _sweep(out, inn, ok, lo, hi, h, last, back, interpolate):
    """One sweep along axis 0 of `out`; `inn` is the input field in the same coordinates, `ok` the lines
    it covers, [lo, hi) its extent along the axis; a backward sweep runs over the flipped axis."""
    if back:
        out, inn = out[::-1], inn[::-1]
        lo, hi = last - hi, last - lo
    for j in range(lo, last - 1):
        covered = ok if j < hi - 1 else np.zeros_like(ok)
        a, b = inn[j], inn[j + 1]
        if interpolate:
            with np.errstate(all="ignore"):
                slope = (b - a) / h
                d = -a / slope
                hit = covered & (a * b <= 0.0) & (np.abs(out[j]) > np.abs(d))
                out[j] = np.where(hit, -d * np.sign(slope), out[j])
        cand = out[j] + np.where(covered, np.sign(b), np.sign(out[j + 1])) * h
        out[j + 1] = np.where(np.abs(cand) < np.abs(out[j + 1]), cand, out[j + 1])


def _redistance(src, sb, ob, h, delta):
    """Signed distance of src (box sb) on the box ob: x and y sweeps per layer, then z sweeps, clamped."""
    n = [ob[a + 3] - ob[a] for a in range(3)]
    lo = [max(sb[a], ob[a]) - ob[a] for a in range(3)]
    hi = [min(sb[a + 3], ob[a + 3]) - ob[a] for a in range(3)]
    out = np.full((n[2], n[1], n[0]), -1.0)
    inn = np.zeros_like(out)
    at = [slice(lo[a] + ob[a] - sb[a], hi[a] + ob[a] - sb[a]) for a in range(3)]
    inn[lo[2]:hi[2], lo[1]:hi[1], lo[0]:hi[0]] = src[at[2], at[1], at[0]]
    k = slice(lo[2], max(lo[2], hi[2] - 1))
    for back in (False, True):  # x: lines are rows from the first covered one on
        o, i = (np.moveaxis(v[k, lo[1]:, :], 2, 0) for v in (out, inn))
        ok = np.broadcast_to(np.arange(lo[1], n[1]) < hi[1], o.shape[1:])
        _sweep(o, i, ok, lo[0], hi[0], h, n[0], back, not back)
    for back in (False, True):  # y
        o, i = (np.moveaxis(v[k, :, lo[0]:], 1, 0) for v in (out, inn))
        ok = np.broadcast_to(np.arange(lo[0], n[0]) < hi[0], o.shape[1:])
        _sweep(o, i, ok, lo[1], hi[1], h, n[1], back, not back)
    o, i = out[:, lo[1]:, lo[0]:], inn[:, lo[1]:, lo[0]:]
    ok = (np.arange(lo[1], n[1]) < hi[1])[:, None] & (np.arange(lo[0], n[0]) < hi[0])[None, :]
    for back in (False, True):  # z
        _sweep(o, i, ok, lo[2], hi[2], h, n[2], back, True)
    return np.clip(out, -delta, delta)


def _cube(b, grid):
    """A box grown to a cube of its longest side, moved back inside [0, grid - 1]."""
    b = list(b)
    side = [b[a + 3] - b[a] for a in range(3)]
    if side[0] == side[1] == side[2]:
        return b
    for a in range(3):
        grow = max(side) - side[a]
        b[a], b[a + 3] = b[a] - grow // 2, b[a + 3] + grow // 2 + grow % 2
    for a in range(3):
        shift = -b[a] if b[a] < 0 else min(0, grid - 1 - b[a + 3])
        b[a], b[a + 3] = b[a] + shift, b[a + 3] + shift
    return b


def _wall_distance(b, p):
    """Distance to the domain wall in voxels; a voxel that no rule covers keeps the one before it."""
    gb, m = p.grid_blowup, p.ngridpoints

    def axis(a):
        c = np.arange(b[a], b[a + 3], dtype=np.float64)
        lo, hi = -(c - gb + 1), c - (m - 1 - gb)
        return np.where(np.abs(lo) < np.abs(hi), lo, hi)

    z, y, x = np.meshgrid(axis(2), axis(1), axis(0), indexing="ij")
    rules = [((x > 0) & (y > 0) & (z > 0), np.sqrt(x * x + y * y + z * z)),
             ((x < 0) & (y < 0) & (z < 0), np.maximum(np.maximum(x, y), z)),
             ((x >= 0) & (y < 0) & (z < 0), x), ((x >= 0) & (y < 0) & (z >= 0), np.sqrt(x * x + z * z)),
             ((x >= 0) & (y >= 0) & (z < 0), np.sqrt(x * x + y * y)),
             ((x < 0) & (y >= 0) & (z < 0), y), ((x < 0) & (y >= 0) & (z >= 0), np.sqrt(y * y + z * z)),
             ((x < 0) & (y < 0) & (z >= 0), z)]
    d = np.select([r[0] for r in rules], [r[1] for r in rules], default=np.nan).ravel()
    known = np.maximum.accumulate(np.where(np.isnan(d), -1, np.arange(d.size)))
    return np.where(known < 0, 0.0, d[np.maximum(known, 0)]).reshape(x.shape)


def _convolve(phi, p):
    n = phi.shape[0]
    k = np.minimum(np.arange(n), n - np.arange(n)).astype(np.float64) ** 2
    s = k[:, None, None] + k[None, :, None] + k[None, None, :n // 2 + 1]
    f = np.exp(-math.sqrt(2 / math.pi) * s * 4.0 * p.dt * p.conv_domain_size ** 2 / (n * n) * math.pi ** 2)
    return np.fft.irfftn(np.fft.rfftn(phi) * f, s=phi.shape, axes=(0, 1, 2))


def _overlap(a, b):
    return [max(a[k], b[k]) for k in range(3)] + [min(a[k + 3], b[k + 3]) for k in range(3)]


def _view(field, box, part):
    return field[part[2] - box[2]:part[5] - box[2], part[1] - box[1]:part[4] - box[1], part[0] - box[0]:part[3] - box[0]]


def exact(case, seed):
    if case["read"] != "fields" or case["physics"] != "none" or voxels(case) * case["steps"] > 1.2e7:
        return None
    p, idfield, bounds, exists = _microstructure(case, seed)
    h, delta, gb, grid = p.h, p.delta, p.grid_blowup, p.ngridpoints
    offsets, ids = G.initial_neighbour_lists(p, bounds, exists)
    alive = [g for g in range(1, case["grains"] + 1) if exists[g]]
    box = {g: _cube([int(v) for v in bounds[g]], grid) for g in alive}
    lists = {g: set(ids[offsets[g]:offsets[g + 1]].tolist()) for g in alive}
    inside = np.zeros(idfield.shape, dtype=bool)
    inside[gb:grid - gb, gb:grid - gb, gb:grid - gb] = True
    phi = {}
    for g in alive:
        b = box[g]
        cut = (slice(b[2], b[5]), slice(b[1], b[4]), slice(b[0], b[3]))
        phi[g] = _redistance(np.where(inside[cut] & (idfield[cut] == g), h, -h), b, b, h, delta)
    for _ in range(case["steps"]):
        field = {g: _convolve(phi[g], p) for g in alive}
        now = set(alive)

        def meets(g, o):
            return all(box[g][a] <= box[o][a + 3] and box[g][a + 3] >= box[o][a] for a in range(3))

        lists.update({g: {o for o in lists[g] if o in now} |
                      {o for nb in lists[g] for o in lists[nb] if o in now and o != g and meets(g, o)} for g in alive})
        compared, grown = {}, {}
        for g in alive:
            b = box[g]
            best = np.full(field[g].shape, -1.0)
            for o in lists[g]:
                part = _overlap(b, box[o])
                if all(part[a] < part[a + 3] for a in range(3)):
                    mine = _view(best, b, part)
                    np.maximum(mine, _view(field[o], box[o], part), out=mine)
            edge, far = gb + p.boundary_grain_tube, grid - gb - p.boundary_grain_tube
            if not (min(b[:3]) > edge and max(b[3:]) < far):
                d = _wall_distance(b, p)
                best = np.where((d > -gb) & (d * h > best), d * h, best)
            v = np.where(np.abs(field[g]) < 0.7 * delta, 0.5 * (field[g] - best), field[g])
            if not (v >= 0).any() or not (v < 0).any():
                continue
            compared[g] = v
            at = np.nonzero(v >= 0)
            lo = [max(0, b[a] + int(at[2 - a].min()) - gb) for a in range(3)]
            hi = [min(grid - 1, b[a] + int(at[2 - a].max()) + gb) for a in range(3)]
            grown[g] = _cube(lo + hi, grid)
        alive = sorted(compared)
        phi = {g: _redistance(compared[g], box[g], grown[g], h, delta) for g in alive}
        box.update(grown)
    return {"phi": _padded((phi[g].ravel() for g in alive), _field_room(case), 0.0, np.float64)}
