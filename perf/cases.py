"""Performance cases of the FIM Eikonal solver: the calls a program makes, over the range of sizes
it makes them at, from a 32 x 32 square (a few microseconds of arithmetic, all latency) to a
96-cells-per-side tetrahedral cube and a batch of 64 solves of uneven cubes.

Every case builds its mesh in numpy (a square split along its cell diagonals, a subdivided
icosahedron, or a cube of six tets per cell whose interior vertices are jittered), hands it to the
library as a user's own mesh, sets speeds or metrics, partitions and uploads it, and then times
one of the library's entry points:

  solve    Mesh.solve: seeds on the host, arrival times back on the host
  noalloc  Mesh.solve_noalloc: seeds and times in device memory, on the program's own stream
  history  Mesh.solve with one launch per outer iteration and the snapshots kept, then the last
           snapshot read
  batch    Batch.solve: many uneven meshes in one launch
  served   Batch with resident meshes: per request a new speed field, sources, and its own times
"""
import functools
import importlib.util
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The repository's Python binding (its folder name holds a hyphen: loaded by path)."""
    if "eikonal_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "eikonal_amd", os.path.join(_ROOT, "sci-solver_eikonal_amd", "eikonal_amd.py"))
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        sys.modules["eikonal_amd"] = mod
    return sys.modules["eikonal_amd"]


# ------------------------------------------------------------------------------------------
# Cases
# ------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call a user makes: the 2D example, one speed, one source in a corner
        dict(name="square32", call="solve", mesh="square", n=32, speed="uniform", sources=1, vpb=64),
        # a small surface inside a GPU pipeline: seeds and times stay on the device
        dict(name="ico5_device", call="noalloc", mesh="ico", n=5, speed="lognormal", sources=2,
             vpb=64),
        # a ragged planar domain of ordinary size with a source set
        dict(name="square301_16src", call="solve", mesh="square", n=301, speed="lognormal",
             sources=16, vpb=64),
        # the anisotropic surface workload: level-7 icosphere, SPD metric per face, 4 sources
        dict(name="ico7_aniso", call="solve", mesh="ico", n=7, speed="metric", sources=4, vpb=64),
        # a large surface: 655,362 vertices, isotropic speeds, one source
        dict(name="ico8_iso", call="solve", mesh="ico", n=8, speed="lognormal", sources=1, vpb=64),
        # a small volume: two layers, several sources
        dict(name="cube16_layers", call="solve", mesh="cube", n=16, speed="layers", sources=5,
             vpb=64),
        # a small ragged volume with a tensor metric per tet, on the device
        dict(name="cube33_tensor", call="noalloc", mesh="cube", n=33, speed="metric", sources=1,
             vpb=64),
        # the main volume workload: 274,625 vertices, 1,572,864 tets, log-normal speeds, centre
        dict(name="cube64", call="solve", mesh="cube", n=64, speed="lognormal", sources=1, vpb=64),
        # the largest single solve: 912,673 vertices, 5.3 million tets, 16 sources
        dict(name="cube96_16src", call="solve", mesh="cube", n=96, speed="lognormal", sources=16,
             vpb=64),
        # the per-iteration history the reference's driver keeps
        dict(name="cube48_history", call="history", mesh="cube", n=48, speed="lognormal",
             sources=1, vpb=64),
        # many uneven volumes at once: 16 cubes of 16..48 cells per side, each with 4 source sets
        dict(name="batch64_cubes", call="batch", mesh="cube", n=16, n_hi=48, meshes=16, sets=4,
             speed="layers", sources=4, vpb=192),
        # requests over resident meshes: 8 slots of a 32^3 cube, 4 of a level-7 icosphere
        dict(name="served12", call="served", mesh="cube", n=32, slots=8, ico=7, ico_slots=4,
             speed="lognormal", sources=6, vpb=192),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case: the same kinds of calls at other sizes, speeds, source counts and block
    sizes (sizes spread over their logarithm)."""
    kind = rng.choice(["square", "square", "ico", "cube", "cube", "cube", "batch", "served"])
    vpb = rng.choice([64, 64, 64, 48, 96, 128])
    sources = _log_int(rng, 1, 64)
    if kind == "square":
        return dict(call=rng.choice(["solve", "noalloc"]), mesh="square",
                    n=_log_int(rng, 20, 600), speed=rng.choice(["uniform", "lognormal", "metric"]),
                    sources=sources, vpb=vpb)
    if kind == "ico":
        return dict(call=rng.choice(["solve", "noalloc"]), mesh="ico", n=rng.choice([4, 5, 6, 7]),
                    speed=rng.choice(["uniform", "lognormal", "metric"]), sources=sources, vpb=vpb)
    if kind == "cube":
        call = rng.choice(["solve", "solve", "noalloc", "history"])
        return dict(call=call, mesh="cube", n=_log_int(rng, 9, 56 if call == "history" else 88),
                    speed=rng.choice(["uniform", "lognormal", "layers", "metric"]), sources=sources,
                    vpb=rng.choice([64, 64, 48, 96]))
    if kind == "batch":
        lo = rng.randint(10, 20)
        return dict(call="batch", mesh="cube", n=lo, n_hi=lo + rng.randint(4, 24),
                    meshes=rng.randint(3, 16), sets=rng.randint(1, 4), speed="layers",
                    sources=rng.randint(1, 8), vpb=rng.choice([64, 128, 192]))
    return dict(call="served", mesh="cube", n=rng.randint(12, 36), slots=rng.randint(1, 8),
                ico=rng.choice([4, 5, 6]), ico_slots=rng.randint(1, 5), speed="lognormal",
                sources=rng.randint(1, 16), vpb=rng.choice([128, 192]))


# ------------------------------------------------------------------------------------------
# Meshes and speeds (numpy)
# ------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _square(n):
    """Unit square, n x n cells split along the (0,0)-(1,1) diagonal."""
    g = (np.arange(n + 1, dtype=np.float64) / n).astype(np.float32)
    xyz = np.zeros(((n + 1) ** 2, 3), np.float32)
    xyz[:, 0] = np.tile(g, n + 1)
    xyz[:, 1] = np.repeat(g, n + 1)
    a = (np.arange(n)[:, None] * (n + 1) + np.arange(n)[None, :]).ravel()
    b, c, d = a + 1, a + n + 1, a + n + 2
    f = np.empty((2 * n * n, 3), np.int32)
    f[0::2] = np.stack([a, b, d], 1)
    f[1::2] = np.stack([a, d, c], 1)
    return xyz, f


@functools.lru_cache(maxsize=6)
def _ico(level):
    """Unit icosphere: an icosahedron whose faces are split in four `level` times."""
    p = (1.0 + 5.0 ** 0.5) / 2.0
    v = np.array([[-1, p, 0], [1, p, 0], [-1, -p, 0], [1, -p, 0], [0, -1, p], [0, 1, p],
                  [0, -1, -p], [0, 1, -p], [p, 0, -1], [p, 0, 1], [-p, 0, -1], [-p, 0, 1]])
    v = v / np.linalg.norm(v, axis=1, keepdims=True)
    # a face for every three corners at the icosahedron's edge length, turned outwards
    near = np.abs(np.linalg.norm(v[:, None] - v[None], axis=2) - np.linalg.norm(v[0] - v[1])) < 1e-9
    f = np.array([(i, j, k) for i in range(12) for j in range(i + 1, 12) for k in range(j + 1, 12)
                  if near[i, j] and near[j, k] and near[i, k]])
    out = np.einsum("ij,ij->i", np.cross(v[f[:, 1]] - v[f[:, 0]], v[f[:, 2]] - v[f[:, 0]]),
                    v[f[:, 0]]) < 0
    f[out] = f[out][:, ::-1]
    for _ in range(level):
        e = np.sort(np.concatenate([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]]), axis=1)
        key, inv = np.unique(e[:, 0].astype(np.int64) * len(v) + e[:, 1], return_inverse=True)
        mid = v[key // len(v)] + v[key % len(v)]
        mid /= np.linalg.norm(mid, axis=1, keepdims=True)
        m = (inv + len(v)).reshape(3, -1)
        ab, bc, ca = m
        f = np.concatenate([np.stack([f[:, 0], ab, ca], 1), np.stack([f[:, 1], bc, ab], 1),
                            np.stack([f[:, 2], ca, bc], 1), np.stack([ab, bc, ca], 1)])
        v = np.concatenate([v, mid])
    return v.astype(np.float32), f.astype(np.int32)


@functools.lru_cache(maxsize=8)
def _cube_tets(n):
    """Six tets per cell, one per order of the axes, along the (0,0,0)-(1,1,1) diagonal."""
    s = n + 1
    k, j, i = np.meshgrid(np.arange(n), np.arange(n), np.arange(n), indexing="ij")
    base = ((k * s + j) * s + i).ravel()
    step = (1, s, s * s)
    cells = []
    for a, b in ((0, 1), (0, 2), (1, 0), (1, 2), (2, 0), (2, 1)):
        p1 = base + step[a]
        p2 = p1 + step[b]
        cells.append(np.stack([base, p1, p2, base + step[0] + step[1] + step[2]], 1))
    return np.stack(cells, 1).reshape(-1, 4).astype(np.int32)


def _cube(n, rng):
    """Unit cube, interior vertices jittered by up to 0.2 of a cell per axis."""
    s = n + 1
    xyz = np.empty((s, s, s, 3))
    g = np.arange(s) / n
    xyz[..., 0], xyz[..., 1], xyz[..., 2] = g[None, None, :], g[None, :, None], g[:, None, None]
    xyz[1:-1, 1:-1, 1:-1] += rng.uniform(-0.2, 0.2, (n - 1, n - 1, n - 1, 3)) / n
    return xyz.reshape(-1, 3).astype(np.float32), _cube_tets(n)


def _rotation(rng, n):
    """n random rotations (unit quaternions)."""
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    w, x, y, z = q.T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)],
                    1).reshape(n, 3, 3)


def _speeds(kind, xyz, elem, rng):
    """What the library's speed call takes for this mesh: tets a factor on the squared lengths
    per tet, or 6 tensor entries; triangles a speed per face, or 3 metric entries; None: speed 1."""
    ne, tet = len(elem), elem.shape[1] == 4
    if kind == "one":
        return None
    if kind == "metric" and tet:
        lam = np.stack([np.ones(ne), rng.uniform(1, 10, ne), rng.uniform(1, 10, ne)], 1)
        r = _rotation(rng, ne)
        m = np.matmul(r * lam[:, None, :], r.transpose(0, 2, 1))
        return m[:, [0, 0, 0, 1, 1, 2], [0, 1, 2, 1, 2, 2]].astype(np.float32)
    if kind == "metric":
        th, k = rng.uniform(0, np.pi, ne), rng.uniform(1, 10, ne)
        c, s = np.cos(th), np.sin(th)
        return np.stack([c * c + k * s * s, (1 - k) * c * s, s * s + k * c * c],
                        1).astype(np.float32)
    if kind == "uniform":
        speed = np.full(ne, rng.uniform(0.5, 2.0))
    elif kind == "layers":
        z = xyz[elem, 2].mean(axis=1)
        speed = np.where(z < rng.uniform(0, 1), 1.0, rng.uniform(0.2, 5.0))
    else:
        speed = np.exp(rng.normal(0.0, 0.5, ne))
    return (1.0 / speed ** 2 if tet else speed).astype(np.float32)


def _mesh_data(kind, n, rng):
    return _square(n) if kind == "square" else _ico(n) if kind == "ico" else _cube(n, rng)


def _problem(case, seed):
    """The inputs of a case as numpy arrays: its meshes (xyz, elements, speed call's values), and
    per solve the mesh it runs on, its sources and, served, its own factors."""
    rng = np.random.default_rng([int(seed), case["n"]])
    meshes, solves = [], []

    def add_mesh(kind, n, speed):
        xyz, elem = _mesh_data(kind, n, rng)
        meshes.append((xyz, elem, _speeds(speed, xyz, elem, rng)))

    def add_solve(i, factors=None):
        solves.append((i, rng.choice(len(meshes[i][0]), case["sources"],
                                     replace=False).astype(np.int32), factors))

    if case["call"] == "batch":
        for i in range(case["meshes"]):
            add_mesh("cube", case["n"] + (i * 7) % (case["n_hi"] - case["n"] + 1), case["speed"])
            for _ in range(case["sets"]):
                add_solve(i)
    elif case["call"] == "served":
        add_mesh("cube", case["n"], "one")
        add_mesh("ico", case["ico"], "one")
        for i, slots in ((0, case["slots"]), (1, case["ico_slots"])):
            for _ in range(slots):
                s = np.exp(rng.normal(0.0, 0.5, len(meshes[i][1])))
                add_solve(i, (1.0 / s ** 2).astype(np.float32))
    else:
        add_mesh(case["mesh"], case["n"], case["speed"])
        add_solve(0)
        if case["sources"] == 1:  # a single source: a corner of the square, the cube's centre
            n = case["n"]
            at = {"square": 0, "cube": ((n // 2) * (n + 1) + n // 2) * (n + 1) + n // 2}
            if case["mesh"] in at:
                solves[0][1][0] = at[case["mesh"]]
    return meshes, solves


# ------------------------------------------------------------------------------------------
# The measured calls
# ------------------------------------------------------------------------------------------
_stream = None


def prepare(case, seed):
    E = _package()
    data, solves = _problem(case, seed)
    meshes = []
    for xyz, elem, values in data:
        tet = elem.shape[1] == 4
        m = E.Mesh.tet(xyz, elem) if tet else E.Mesh.tri(xyz, elem)
        if values is not None and not tet and values.ndim == 2:
            m.set_metric_tri(values)
        elif values is not None:
            m.set_speed(values)
        m.partition(case["vpb"])
        meshes.append(m)
    state = dict(call=case["call"], meshes=meshes, seeds=[s for _, s, _ in solves])
    if case["call"] in ("batch", "served"):
        state["batch"] = E.Batch([meshes[i] for i, _, _ in solves])
        if case["call"] == "served":
            # a request's speed field lies in pinned memory, as a server receives it
            state["factors"] = [torch.from_numpy(f).pin_memory().numpy() for _, _, f in solves]
        return state
    meshes[0].upload()
    if case["call"] == "noalloc":
        global _stream
        if _stream is None:
            _stream = torch.cuda.Stream()
        state["dev_seeds"] = torch.from_numpy(state["seeds"][0]).cuda()
        state["dev_out"] = torch.empty(len(data[0][0]), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    return state


def run(state):
    call = state["call"]
    if call == "noalloc":
        # the calls of one device share the library's scratch array: one stream for all of them
        state["meshes"][0].solve_noalloc(state["dev_seeds"].data_ptr(), state["dev_seeds"].numel(),
                                         state["dev_out"].data_ptr(), _stream.cuda_stream)
        return state["dev_out"]
    if call == "solve":
        return state["meshes"][0].solve(state["seeds"][0])[0]
    if call == "history":
        E, m = _package(), state["meshes"][0]
        t, st = m.solve(state["seeds"][0], scheduler=E.SCHED_SYNC, record_history=1)
        return {"times": t, "last": m.history(st["history_len"] - 1)}
    b = state["batch"]
    if call == "batch":
        return b.solve(state["seeds"], max_inner=1)[0]
    for i, f in enumerate(state["factors"]):
        b.set_factors(i, f)
    b.solve(state["seeds"], out=False, max_inner=1)
    return [b.result(i) for i in range(len(state["seeds"]))]


def _counts(case):
    """(vertices, elements, corners) of every solve of a case."""
    def one(kind, n):
        if kind == "square":
            return (n + 1) ** 2, 2 * n * n, 3
        if kind == "ico":
            return 10 * 4 ** n + 2, 20 * 4 ** n, 3
        return (n + 1) ** 3, 6 * n ** 3, 4
    if case["call"] == "batch":
        return [one("cube", case["n"] + (i * 7) % (case["n_hi"] - case["n"] + 1))
                for i in range(case["meshes"]) for _ in range(case["sets"])]
    if case["call"] == "served":
        return [one("cube", case["n"])] * case["slots"] + [one("ico", case["ico"])] * case["ico_slots"]
    return [one(case["mesh"], case["n"])]


def work(case):
    """Per element its corner ids and metric values (6 per tet, 3 per triangle) once, its corners
    solved once (about 150 operations per tet corner, 40 per triangle corner); per vertex its time
    written once; served: the factors; history: the last snapshot."""
    b = f = 0
    for nv, ne, k in _counts(case):
        b += ne * (4 * k + (24 if k == 4 else 12)) + 4 * nv
        f += ne * (4 * 150 if k == 4 else 3 * 40)
        b += 4 * ne if case["call"] == "served" else 4 * nv if case["call"] == "history" else 0
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------------------------------
# The same results in 64 bits
# ------------------------------------------------------------------------------------------
def _right_angle_faces(xyz, f):
    """The square's virtual faces.  A corner whose angle, evaluated in single precision, is not
    below a right angle is split by the diagonal to the far corner of the face across its
    opposite edge; each half updates that corner only.  Returns (faces, their origins)."""
    p = xyz[f]  # float32, as the rule is stated on them
    rows, origin = [], []
    across = np.empty(len(f), np.int64)
    across[0::2], across[1::2] = f[1::2, 2], f[0::2, 1]  # far corner beyond the cell's diagonal
    for k in range(3):
        d = lambda i, j: np.sqrt(((p[:, i] - p[:, j]) ** 2).astype(np.float32).sum(1, dtype=np.float32))  # noqa: E731
        i, j = (k + 1) % 3, (k + 2) % 3
        a, b, c = d(i, j), d(k, j), d(k, i)
        x = (b * b + c * c - a * a) / (2 * b * c)
        wide = np.nonzero(np.arccos(x, dtype=np.float32).astype(np.float64) >= np.pi / 2)[0]
        v, v2, v4, v3 = f[wide, k], f[wide, i], f[wide, j], across[wide]
        rows += [np.stack([v, v2, v3], 1), np.stack([v, v3, v4], 1)]
        origin += [wide, wide]
    return np.concatenate(rows), np.concatenate(origin)


def _edges2(xyz, elem, values, factors, pairs, origin=None, frame=None):
    """Squared metric lengths of the given corner pairs, float64 [elements, pairs]."""
    p = xyz[elem].astype(np.float64)
    d = np.stack([p[:, b] - p[:, a] for a, b in pairs], 1)
    v = None if values is None else values[origin if origin is not None else slice(None)].astype(np.float64)
    if v is not None and v.ndim == 2 and elem.shape[1] == 4:
        q = (v[:, None, 0] * d[..., 0] ** 2 + v[:, None, 3] * d[..., 1] ** 2 +
             v[:, None, 5] * d[..., 2] ** 2 + 2 * (v[:, None, 1] * d[..., 0] * d[..., 1] +
             v[:, None, 2] * d[..., 0] * d[..., 2] + v[:, None, 4] * d[..., 1] * d[..., 2]))
    elif v is not None and v.ndim == 2:
        # the metric's frame: along the face's first edge, and across it in the face's plane
        o = xyz[frame if frame is not None else elem].astype(np.float64)
        e1, e2 = o[:, 1] - o[:, 0], o[:, 2] - o[:, 0]
        t1 = e1 / np.linalg.norm(e1, axis=1, keepdims=True)
        t2 = e2 - (e2 * t1).sum(1, keepdims=True) * t1
        t2 /= np.linalg.norm(t2, axis=1, keepdims=True)
        x, y = (d * t1[:, None]).sum(2), (d * t2[:, None]).sum(2)
        q = x * x * v[:, None, 0] + 2 * x * y * v[:, None, 1] + y * y * v[:, None, 2]
    else:
        q = (d ** 2).sum(2)
        if v is not None:
            q = q * (v[:, None] if elem.shape[1] == 4 else 1 / v[:, None] ** 2)
    return q if factors is None else q * factors.astype(np.float64)[:, None]


_PAIRS = {4: ((0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)), 3: ((0, 1), (0, 2), (1, 2))}


def _two(a, b, la, lb, lab):
    """Least cost through the inside of the segment between two corners: times a, b >= 0, squared
    lengths la, lb to the target and lab between them; inf where the minimum is at an end."""
    g = 0.5 * (la + lb - lab)
    ra, rb = lb - g, la - g
    wa, wb = lb * a - g * b, la * b - g * a
    A, B, C = ra + rb, wa + wb, a * wa + b * wb - (la * lb - g * g)
    disc = B * B - A * C
    d = (B + disc.clamp(min=0).sqrt()) / A
    x, y = d * ra - wa, d * rb - wb
    s = x + y
    t = (x * a + y * b + ((x * la + y * lb) * s - x * y * lab).clamp(min=0).sqrt()) / s
    return torch.where((disc >= 0) & (x >= 0) & (y >= 0) & (s > 0), t, torch.inf)


def _three(a, b, c, la, lb, lc, lab, lac, lbc):
    """The same through the inside of a triangle of three corners."""
    gab, gac, gbc = 0.5 * (la + lb - lab), 0.5 * (la + lc - lac), 0.5 * (lb + lc - lbc)
    kaa, kbb, kcc = lb * lc - gbc * gbc, la * lc - gac * gac, la * lb - gab * gab
    kab, kac, kbc = gac * gbc - gab * lc, gab * gbc - gac * lb, gab * gac - la * gbc
    ra, rb, rc = kaa + kab + kac, kab + kbb + kbc, kac + kbc + kcc
    wa, wb, wc = kaa * a + kab * b + kac * c, kab * a + kbb * b + kbc * c, kac * a + kbc * b + kcc * c
    A, B = ra + rb + rc, wa + wb + wc
    C = a * wa + b * wb + c * wc - (la * kaa + gab * kab + gac * kac)
    disc = B * B - A * C
    d = (B + disc.clamp(min=0).sqrt()) / A
    x, y, z = d * ra - wa, d * rb - wb, d * rc - wc
    s = x + y + z
    q = (x * la + y * lb + z * lc) * s - x * y * lab - x * z * lac - y * z * lbc
    t = (x * a + y * b + z * c + q.clamp(min=0).sqrt()) / s
    return torch.where((disc >= 0) & (x >= 0) & (y >= 0) & (z >= 0) & (s > 0), t, torch.inf)


def _corner(c, t, length):
    """Least arrival at corner c of elements with corner times t (a list) from the others."""
    others = [i for i in range(len(t)) if i != c]
    known = {i: torch.isfinite(t[i]) for i in others}
    t0 = torch.stack([t[i] for i in others]).amin(0)
    tau = {i: torch.where(known[i], t[i] - t0, 0.0) for i in others}
    best = torch.stack([torch.where(known[i], tau[i] + length(c, i).sqrt(), torch.inf)
                        for i in others]).amin(0)
    for k, i in enumerate(others):
        for j in others[k + 1:]:
            v = _two(tau[i], tau[j], length(c, i), length(c, j), length(i, j))
            best = torch.minimum(best, torch.where(known[i] & known[j], v, torch.inf))
    if len(others) == 3:
        i, j, k = others
        v = _three(tau[i], tau[j], tau[k], length(c, i), length(c, j), length(c, k), length(i, j),
                   length(i, k), length(j, k))
        best = torch.minimum(best, torch.where(known[i] & known[j] & known[k], v, torch.inf))
    return t0 + best


def _fixed_point(nv, groups, sources):
    """Arrival times of the sources over element groups (elements, squared lengths, corners that
    are updated): every element around a changed vertex is solved again until none changes."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    groups = [(torch.from_numpy(e.astype(np.int64)).to(dev), torch.from_numpy(q).to(dev), k)
              for e, q, k in groups]
    T = torch.full((nv,), torch.inf, dtype=torch.float64, device=dev)
    T[torch.from_numpy(sources).to(dev).long()] = 0.0
    changed = torch.isfinite(T)
    while bool(changed.any()):
        before = T.clone()
        for elem, q, corners in groups:
            act = torch.nonzero(changed[elem].any(1)).ravel()
            for part in act.split(4_000_000):
                e, l2 = elem[part], q[part]
                pair = {p: l2[:, i] for i, p in enumerate(_PAIRS[e.shape[1]])}
                t = [before[e[:, k]] for k in range(e.shape[1])]
                for c in range(corners):
                    new = _corner(c, t, lambda a, b: pair[min(a, b), max(a, b)])
                    T.scatter_reduce_(0, e[:, c], new.nan_to_num(torch.inf, torch.inf), "amin")
        changed = T < before * (1 - 1e-13)
        changed |= torch.isfinite(T) & ~torch.isfinite(before)
    return T.cpu().numpy()


def exact(case, seed):
    meshes, solves = _problem(case, seed)
    # all solves of the case side by side, as one disconnected problem per element kind
    out = [None] * len(solves)
    for k in (3, 4):
        base, parts, virt, src, where = 0, [], [], [], []
        for n, (i, seeds, factors) in enumerate(solves):
            xyz, elem, values = meshes[i]
            if elem.shape[1] != k:
                continue
            parts.append((elem + base, _edges2(xyz, elem, values, factors, _PAIRS[k])))
            if case["mesh"] == "square" and k == 3:
                f, origin = _right_angle_faces(xyz, elem)
                virt.append((f + base, _edges2(xyz, f, values, None, _PAIRS[3], origin, elem[origin])))
            src.append(seeds.astype(np.int64) + base)
            where.append((n, base, len(xyz)))
            base += len(xyz)
        if not parts:
            continue
        groups = [(np.concatenate([e for e, _ in parts]), np.concatenate([q for _, q in parts]), k)]
        if virt and sum(len(e) for e, _ in virt):
            groups.append((np.concatenate([e for e, _ in virt]),
                           np.concatenate([q for _, q in virt]), 1))
        T = _fixed_point(base, groups, np.concatenate(src))
        for n, b, nv in where:
            out[n] = T[b:b + nv]
    if case["call"] in ("batch", "served"):
        return out
    return {"times": out[0], "last": out[0]} if case["call"] == "history" else out[0]
