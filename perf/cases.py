"""Performance cases of the boolean hot path: the calls that programs built on
this package make, over the sizes its tests, its benchmark and its users have.

Meshes are closed: subdivided icospheres (sculpted parts, the benchmark's
shape), tori of any odd resolution (ragged sizes) and gridded cubes that nearly
share faces (CAD parts).  A case's "kind" is the way the package is called:

  pair        meshes resident on the GPU, one boolean hot path per pass:
              prepare both, candidate pairs, triangle-triangle tests, the
              intersecting pairs and segments, both meshes' votes
  host_pair   the same from host arrays, the meshes created in the pass
  batch       many small pairs in one captured run: counts and sides
  frame       a batch animated: new coordinates, run, candidates and sides
  points      inside/outside of points against one prepared mesh
  tri_tri     the triangle-triangle test on a caller's own pair list
  components  face groups of one mesh, a band of triangles blocked
  adjoint     forward and backward of the differentiable boolean
  combine     the whole boolean through the drop-in classes
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from solidboolean_amd import diff, dropin, meshgen as mg, native as N

PRECISION = {"fp64": N.FP64, "filtered": N.FP32_FILTERED}


def listed():
    return [
        # two 80-triangle meshes: launch and call latency is all there is
        dict(name="pair_sphere_80", kind="pair", shape="sphere", size=1, precision="filtered"),
        # an ordinary part: 81,920 triangles each
        dict(name="pair_sphere_82k", kind="pair", shape="sphere", size=6, precision="filtered"),
        # the benchmark's pair: 1,310,720 triangles each, rough surfaces
        dict(name="pair_sphere_1311k", kind="pair", shape="sphere", size=8, precision="filtered"),
        # faces 1e-6 apart over half of each cube, plain FP64 throughout
        dict(name="pair_cube_393k_fp64", kind="pair", shape="cube", size=181, precision="fp64"),
        # a dense scan against a small tool, straight from host arrays
        dict(name="host_torus_543k", kind="host_pair", shape="torus", size=387, precision="filtered"),
        # thousands of small independent booleans
        dict(name="batch_4096", kind="batch", pairs=4096, precision="filtered"),
        # an animated scene: the vertices change every frame
        dict(name="frame_97_fp64", kind="frame", pairs=97, precision="fp64"),
        # point-in-solid queries with the three rays' answers
        dict(name="points_100k", kind="points", shape="sphere", size=6, points=100003, axes=True,
             precision="filtered"),
        # a caller's own candidate pairs
        dict(name="tri_tri_65k", kind="tri_tri", pairs=65521),
        # face groups of a dense mesh
        dict(name="components_1311k", kind="components", shape="torus", size=603),
        # one optimisation step through a union
        dict(name="adjoint_20k", kind="adjoint", size=5, op="union"),
        # a whole boolean as a user of the classes makes it
        dict(name="combine_20k", kind="combine", size=5, robust=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair", "pair", "pair", "host_pair", "batch", "frame", "points", "tri_tri", "components",
                       "adjoint", "combine"])
    precision = rng.choice(["filtered", "filtered", "fp64"])
    if kind in ("pair", "host_pair"):
        shape = rng.choice(["sphere", "torus", "torus", "cube"])
        size = {"sphere": lambda: rng.randint(1, 7), "torus": lambda: _log_int(rng, 5, 600),
                "cube": lambda: _log_int(rng, 2, 300)}[shape]()
        return dict(kind=kind, shape=shape, size=size, precision=precision)
    if kind == "batch":
        return dict(kind=kind, pairs=_log_int(rng, 8, 4000), precision=precision)
    if kind == "frame":
        return dict(kind=kind, pairs=_log_int(rng, 1, 512), precision=precision)
    if kind == "points":
        return dict(kind=kind, shape=rng.choice(["sphere", "torus"]), size=rng.randint(3, 6),
                    points=_log_int(rng, 24, 400000), axes=rng.random() < 0.5, precision=precision)
    if kind == "tri_tri":
        return dict(kind=kind, pairs=_log_int(rng, 2, 100000))
    if kind == "components":
        return dict(kind=kind, shape="torus", size=_log_int(rng, 5, 600))
    if kind == "adjoint":
        return dict(kind=kind, size=rng.randint(2, 5), op=rng.choice(["union", "diff", "intersect"]))
    return dict(kind=kind, size=rng.randint(2, 5), robust=rng.random() < 0.3)


# --- inputs -----------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _sphere(level):
    return mg.icosphere(level)


def _torus_counts(size):
    """Segments around the axis and around the tube (both odd or ragged)."""
    return 2 * size - size // 5 + 4, size


def _counts(shape, size):
    """(vertices, triangles) of one mesh."""
    if shape == "sphere":
        return 10 * 4 ** size + 2, 20 * 4 ** size
    if shape == "torus":
        nu, nv = _torus_counts(size)
        return nu * nv, 2 * nu * nv
    return 6 * size * size + 2, 12 * size * size


def _tool_size(size):
    """The second torus of a pair: a fifth of the first one's resolution."""
    return max(3, size // 5)


def _moved(mesh, stream, offset):
    shift = [o + 0.02 * float(u) for o, u in zip(offset, 2.0 * stream.uniform(3) - 1.0)]
    return mg.transform(mesh, mg.random_rotation(stream), shift)


# How two meshes lie to each other belongs to the case (so that every seed has
# as many intersecting pairs); the seed places the two together in space and
# orders their triangles.
def _relabel(mesh, stream):
    """The triangle list from another start on."""
    return mg.Mesh(mesh.vertices, np.roll(mesh.triangles, int(stream.next_u64(1)[0] % np.uint64(mesh.nt)), axis=0))


def _placed(meshes, stream):
    """Rotated and shifted together."""
    rot, shift = mg.random_rotation(stream), 0.3 * (2.0 * stream.uniform(3) - 1.0)
    return [mg.transform(m, rot, shift) for m in meshes]


def _turned(meshes, stream):
    """Turned together by half turns about the axes, every rounding the same:
    for meshes whose exact ties, candidates or welds a rotation would change."""
    k = int(stream.next_u64(1)[0] % np.uint64(3))
    sign = np.array([1.0 if axis == k else -1.0 for axis in range(3)])
    return [mg.Mesh(m.vertices * sign, m.triangles) for m in meshes]


def _pair(shape, size, seed):
    stream, place = mg.SplitMix64(size * 7919 + 12345), mg.SplitMix64(seed * 7919 + 1)
    if shape == "cube":
        a = mg.cube_grid(size)
        pair = _turned([a, mg.transform(a, None, (1e-6, 0.5, 0.5))], place)
    elif shape == "torus":
        a = mg.radial_noise(mg.torus(1.0, 0.3, *_torus_counts(size)), 1e-4, stream)
        b = mg.radial_noise(mg.torus(0.5, 0.2, *_torus_counts(_tool_size(size))), 1e-4, stream)
        pair = _placed([a, _moved(b, stream, (0.7, 0.3, 0.1))], place)
    else:
        a = mg.radial_noise(_sphere(size), 1e-3, stream)
        b = mg.radial_noise(_sphere(size), 1e-3, stream)
        pair = _placed([a, _moved(b, stream, (0.4, 0.25, 0.1))], place)
    return [_relabel(m, place) for m in pair]


def _smooth_pair(level, seed):
    """Smooth spheres, as the whole-boolean tests use them."""
    place = mg.SplitMix64(seed * 104729 + 77)
    pair = [_sphere(level), _moved(_sphere(level), mg.SplitMix64(level + 40), (0.5, 0.3, 0.2))]
    return [_relabel(m, place) for m in _turned(pair, place)]


def _many_pairs(npairs, seed, moved):
    """Sphere pairs of uneven sizes as mg.batch_pairs makes them, each pair
    placed by the seed: anywhere (moved), or by half turns."""
    place = mg.SplitMix64(seed * 65537 + 3)
    out = []
    for pair in mg.batch_pairs(npairs, npairs + 1):
        out.append(tuple(_placed(pair, place) if moved else _turned(pair, place)))
    return out


_contexts = {}


def _context(precision):
    """The program's context (one per ray precision, kept like a device handle)."""
    if precision not in _contexts:
        _contexts[precision] = N.Context(0)
        _contexts[precision].set_tuning(ray_precision=PRECISION[precision])
    return _contexts[precision]


def prepare(case, seed):
    kind = case["kind"]
    precision = case.get("precision", "filtered")
    ctx = _context(precision)
    state = dict(case=case, ctx=ctx, precision=PRECISION[precision])
    if kind in ("pair", "host_pair"):
        a, b = _pair(case["shape"], case["size"], seed)
        # page-locked vote arrays, kept from pass to pass
        state["votes"] = (N.host_array(a.nt), N.host_array(b.nt))
        if kind == "pair":
            state["A"] = ctx.mesh(a.vertices, a.triangles, prepare=False)
            state["B"] = ctx.mesh(b.vertices, b.triangles, prepare=False)
        else:
            state["a"], state["b"] = a, b
    elif kind in ("batch", "frame"):
        pairs = _many_pairs(case["pairs"], seed, kind == "batch")
        state["batch"] = ctx.batch(pairs)
        state["batch"].run(state["precision"])  # sizes its buffers and captures its graph, once per shape
        if kind == "frame":  # the next frame: the scene at half its size
            state["xyz"] = 0.5 * np.concatenate([m.vertices for p in pairs for m in p])
    elif kind == "points":
        a = _pair(case["shape"], case["size"] if case["shape"] == "sphere" else 5 << case["size"], seed)[0]
        stream = mg.SplitMix64(seed * 31 + 5)
        state["A"] = ctx.mesh(a.vertices, a.triangles)
        state["points"] = 1.1 * (2.0 * stream.uniform(3 * case["points"]) - 1.0).reshape(-1, 3)
    elif kind == "tri_tri":
        stream = mg.SplitMix64(seed * 13 + 3)
        n = case["pairs"]
        state["a9"] = stream.uniform(9 * n).reshape(n, 9)
        state["b9"] = stream.uniform(9 * n).reshape(n, 9)
    elif kind == "components":
        a = _pair(case["shape"], case["size"], seed)[0]
        stream = mg.SplitMix64(seed + 99)
        state["A"] = ctx.mesh(a.vertices, a.triangles, prepare=False)
        # a run of neighbouring triangles (cut ones) and a few loose ones
        state["blocked"] = (stream.uniform(a.nt) < 1e-3).astype(np.uint8)
        state["blocked"][a.nt // 3: a.nt // 3 + max(1, int(0.02 * float(stream.uniform(1)[0]) * a.nt))] = 1
    elif kind == "adjoint":
        a, b = _smooth_pair(case["size"], seed)
        state["topology"] = diff.Topology(a.vertices, a.triangles, b.vertices, b.triangles, case["op"])
        stream = mg.SplitMix64(seed + 5)
        # some optimisation steps later
        xyz = state["topology"].input_xyz
        state["xyz"] = torch.from_numpy(xyz + 1e-5 * (2.0 * stream.uniform(xyz.size).reshape(-1, 3) - 1.0))
        state["weight"] = torch.from_numpy(stream.uniform(3 * state["topology"].nderived).reshape(-1, 3))
    else:
        state["a"], state["b"] = _smooth_pair(case["size"], seed)
    return state


# --- one pass ---------------------------------------------------------------
def _boolean(state, A, B):
    A.prepare()
    B.prepare()
    P = A.find_pairs(B)
    P.tri_tri(A, B, state["precision"], stats=False)
    pairs, segments = P.hits()
    va, vb = A.classify_pair(B, P, out=state["votes"])
    return dict(pairs=pairs, segments=segments, votes_a=va, votes_b=vb)


def run(state):
    kind, ctx = state["case"]["kind"], state["ctx"]
    if kind == "pair":
        return _boolean(state, state["A"], state["B"])
    if kind == "host_pair":
        a, b = state["a"], state["b"]
        return _boolean(state, ctx.mesh(a.vertices, a.triangles, prepare=False),
                        ctx.mesh(b.vertices, b.triangles, prepare=False))
    if kind == "batch":
        state["batch"].run(state["precision"])
        candidates, hits = state["batch"].counts()
        return dict(candidates=candidates, hits=hits, sides=state["batch"].sides())
    if kind == "frame":
        state["batch"].set_vertices(state["xyz"])
        state["batch"].run(state["precision"])
        pairs, status, segments = state["batch"].candidates()
        return dict(pairs=pairs, status=status, segments=segments, sides=state["batch"].sides())
    if kind == "points":
        axes, inside = state["A"].classify_points(state["points"])
        return dict(axes=axes, inside=inside) if state["case"]["axes"] else inside
    if kind == "tri_tri":
        status, segments = ctx.tri_tri_batch(state["a9"], state["b9"])
        return dict(status=status, segments=segments)
    if kind == "components":
        return state["A"].components(state["blocked"])
    if kind == "adjoint":
        xyz = state["xyz"].detach().requires_grad_(True)
        volume, derived = diff.volume_and_vertices(xyz, state["topology"], ctx)
        (volume + (derived * state["weight"]).sum()).backward()
        return dict(volume=volume.detach(), derived=derived.detach(), grad=xyz.grad)
    a, b = state["a"], state["b"]
    A, B = dropin.SolidMesh(a.vertices, a.triangles), dropin.SolidMesh(b.vertices, b.triangles)
    A.prepare()
    B.prepare()
    sb = dropin.SolidBoolean(A, B, robust_weld=state["case"]["robust"])
    if not sb.combine():
        return dict(ok=False)
    return dict(ok=True, vertices=sb.result_vertices(), union=sb.fetch_union(), difference=sb.fetch_diff(),
                intersection=sb.fetch_intersect())


# --- what a pass needs, and what it may differ by ---------------------------
def work(case):
    """Inputs read once and outputs written once.  Operations: per triangle its
    normal and box (about 60) and two rays with one tested candidate each
    (about 120); per triangle pair the two planes' signs (about 80)."""
    kind = case["kind"]
    if kind in ("pair", "host_pair", "combine"):
        shape = case.get("shape", "sphere")
        va, ta = _counts(shape, case["size"])
        vb, tb = _counts(shape, _tool_size(case["size"]) if shape == "torus" else case["size"])
        index = 12 if kind == "pair" else 24
        out = ta + tb if kind != "combine" else 24 * (va + vb) + 2 * 24 * (ta + tb)
        return dict(bytes=24 * (va + vb) + index * (ta + tb) + out, flops=180 * (ta + tb))
    if kind in ("batch", "frame"):
        p = np.array([4.0 ** -l for l in mg.BATCH_LEVELS])
        p /= p.sum()
        nt = 2 * case["pairs"] * float(sum(q * 20 * 4 ** l for q, l in zip(p, mg.BATCH_LEVELS)))
        nv = nt / 2 + 4 * case["pairs"]
        # about 0.38 candidates per triangle on these pairs (8 B, a status byte and a segment each)
        out = nt + (0.38 * 57 * nt if kind == "frame" else 0)
        return dict(bytes=int(24 * nv + 12 * nt + out), flops=int(180 * nt))
    if kind == "points":
        n = case["points"]
        return dict(bytes=24 * n + n * (4 if case["axes"] else 1), flops=60 * n * (3 if case["axes"] else 2))
    if kind == "tri_tri":
        return dict(bytes=case["pairs"] * (144 + 1 + 48), flops=80 * case["pairs"])
    if kind == "components":
        nt = _counts(case["shape"], case["size"])[1]
        return dict(bytes=17 * nt, flops=3 * nt)
    # adjoint: inputs, faces (about as many as both inputs hold), derived vertices along the curve, gradient
    nv, nt = _counts("sphere", case["size"])
    nd = 12 * 2 ** case["size"]
    return dict(bytes=2 * nv * 48 + 2 * nt * 12 + nd * (20 + 24), flops=60 * 2 * nt + 300 * nd)


def tolerance(case):
    if case["kind"] == "adjoint":
        # sums over a vertex's faces in FP64, in an order that varies from run
        # to run: 4.3e-16 and 3.5e-15 between two runs (1.1e-16 from the exact
        # gradient), with room for more faces and a steeper crossing
        return {"rel": 4e-15, "max": 4e-14}
    return "exact"


# --- 64-bit values in plain numpy -------------------------------------------
def _cross(a, b):
    return np.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                     a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], 1)


def _dot(a, b):
    return (a * b).sum(1)


def _exact_tri_tri(a9, b9):
    """Segments of the intersecting pairs: both triangles' spans on the line the
    planes share; zero elsewhere."""
    A, B = a9.astype(np.longdouble).reshape(-1, 3, 3), b9.astype(np.longdouble).reshape(-1, 3, 3)
    na = _cross(A[:, 1] - A[:, 0], A[:, 2] - A[:, 0])
    nb = _cross(B[:, 0] - B[:, 2], B[:, 1] - B[:, 2])
    line = _cross(na, nb)

    def span(tri, normal, point):
        """The tri's two edge crossings of the plane in order along the line
        (parameter, point), and whether one of its vertices is alone above."""
        d = np.stack([_dot(tri[:, k] - point, normal) for k in range(3)], 1)
        crosses = (d.min(1) < 0) & (d.max(1) > 0)
        pos = np.full((len(tri), 2), np.inf, np.longdouble)
        pts = np.zeros((len(tri), 2, 3), np.longdouble)
        found = np.zeros(len(tri), int)
        for k in range(3):
            i, j = k, (k + 1) % 3
            hit = ((d[:, i] > 0) != (d[:, j] > 0)) & crosses & (found < 2)
            r = np.nonzero(hit)[0]
            t = d[r, i] / (d[r, i] - d[r, j])
            x = tri[r, i] + t[:, None] * (tri[r, j] - tri[r, i])
            pts[r, found[r]] = x
            pos[r, found[r]] = _dot(x, line[r])
            found[r] += 1
        order = pos[:, 0] > pos[:, 1]
        pos[order] = pos[order][:, ::-1]
        pts[order] = pts[order][:, ::-1]
        return crosses, pos, pts, (d > 0).sum(1) == 1

    ca, pa, xa, alone_a = span(A, nb, B[:, 2])
    cb, pb, xb, alone_b = span(B, na, A[:, 0])
    lo_a, hi_a = pa[:, 0] > pb[:, 0], pa[:, 1] < pb[:, 1]
    lo = np.where(lo_a[:, None], xa[:, 0], xb[:, 0])
    hi = np.where(hi_a[:, None], xa[:, 1], xb[:, 1])
    hit = ca & cb & (np.maximum(pa[:, 0], pb[:, 0]) <= np.minimum(pa[:, 1], pb[:, 1]))
    hi_first = (alone_a != alone_b)[:, None]
    seg = np.concatenate([np.where(hi_first, hi, lo), np.where(hi_first, lo, hi)], 1)
    return np.where(hit[:, None], seg, 0).astype(np.float64)


def _exact_adjoint(xyz, src, faces, weight):
    x, y = xyz[src[:, 0]], xyz[src[:, 1]]
    p0, p1, p2 = xyz[src[:, 2]], xyz[src[:, 3]], xyz[src[:, 4]]
    e, w, c, d = y - x, p0 - x, p2 - p0, p1 - p0
    n = _cross(d, c)
    b = _dot(e, n)
    t = _dot(w, n) / b
    derived = x + t[:, None] * e
    every = np.concatenate([xyz, derived])
    f0, f1, f2 = every[faces[:, 0]], every[faces[:, 1]], every[faces[:, 2]]
    volume = math.fsum(_dot(f0, _cross(f1, f2)) / 6.0)
    grad = np.zeros_like(every)
    for k, g in ((0, _cross(f1, f2)), (1, _cross(f2, f0)), (2, _cross(f0, f1))):
        np.add.at(grad, faces[:, k], g / 6.0)
    g = grad[len(xyz):] + weight
    s = _dot(g, e) / b
    m = w - t[:, None] * e
    along = g - s[:, None] * n
    g1, g2 = s[:, None] * _cross(c, m), s[:, None] * _cross(m, d)
    out = grad[:len(xyz)]
    for k, v in ((0, (1.0 - t)[:, None] * along), (1, t[:, None] * along), (2, s[:, None] * n - g1 - g2),
                 (3, g1), (4, g2)):
        np.add.at(out, src[:, k], v)
    return volume, derived, out


def exact(case, seed):
    """Values in 64 bits or better; None for flags, indices and for segments
    whose pairs only a whole search gives."""
    if case["kind"] == "tri_tri":
        stream = mg.SplitMix64(seed * 13 + 3)
        n = case["pairs"]
        a9, b9 = stream.uniform(9 * n).reshape(n, 9), stream.uniform(9 * n).reshape(n, 9)
        return dict(status=None, segments=_exact_tri_tri(a9, b9))
    if case["kind"] == "adjoint":
        state = prepare(case, seed)
        topo = state["topology"]
        volume, derived, grad = _exact_adjoint(state["xyz"].numpy(), topo.src.astype(np.int64), topo.faces.astype(np.int64),
                                               state["weight"].numpy())
        return dict(volume=np.float64(volume), derived=derived, grad=grad)
    return None
