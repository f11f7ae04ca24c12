"""The work that users of the MCUT front end have it do, as timed cases.

``listed()`` gives the cases, ``draw(rng)`` one more of the same ranges,
``prepare(case, seed)`` what a program has in hand before the call, ``run``
one pass through the public entry points (mcut_amd.frontend) with its
outputs, ``work`` the bytes and operations a pass cannot do without, and
``exact`` the outputs from plain numpy in 64 bits.

A case's ``kind`` says which entry points it takes:

- ``device``: one source/cut pair already in GPU memory, the registry left
  there (``Context.dispatch_device`` and the registry's device pointers);
- ``host``: host meshes in, registry read back (``Context.dispatch``), one
  pair after another through one context;
- ``retry``: a dispatch that violates general position and its rerun with a
  perturbed cut mesh (``Context.redispatch_perturbed``);
- ``cutpath``: a dispatch and the cut-path edges made from its registry;
- ``seam``: the two calls MCUT itself makes when it runs on this library,
  ``Context.broad_phase`` over its face boxes and ``Context.dispatch_narrow``
  on its shifted meshes and those pairs;
- ``batch``: many pairs in one ``Context.dispatch_batch_device``;
- ``serve``: one resident source mesh and a burst of cut requests
  (``Server.run``).

A program keeps its context (or server) and brings new meshes to it, so the
handle outlives a state; it is made anew when another case begins.
"""
import functools
import math

import numpy as np
import torch

from mcut_amd import frontend as fe
from mcut_amd import meshgen as mg

_U32 = np.uint32


def listed():
    return [
        # the smallest calls: a 960-triangle sphere cut by a 192-triangle cube
        # (the size of the reference's own examples); latency and launches count
        {"name": "pair_small", "kind": "device", "shape": "uv", "n": 32, "m": 4},
        # polygon meshes from a modeller, as host arrays: a box of quads cut by
        # a prism with 24-gon caps, registry read back
        {"name": "polygons_host", "kind": "host", "shape": "polygon", "n": 30, "m": 24, "count": 1},
        # a program that cuts pairs of uneven size one after another: spheres of
        # 200-200k triangles against boxes of 12-12k, host arrays, registry read back
        {"name": "pairs_mixed_host", "kind": "host", "shape": "mix", "n": 100, "m": 32, "count": 16},
        # the repository's headline pair: two subdivision-7 icospheres, resident
        {"name": "pair_ico7", "kind": "device", "shape": "ico", "n": 7, "m": 7},
        # the largest single pair: two spheres of 1.3 M triangles
        {"name": "pair_ico8", "kind": "device", "shape": "ico", "n": 8, "m": 8},
        # degenerate-heavy sectioning: a 2 M-triangle terrain, many vertices
        # exactly on the cut plane, millions of tests
        {"name": "terrain", "kind": "device", "shape": "terrain", "n": 1024, "m": 64},
        # general position violated (a sphere vertex on the cube's face), then
        # the rerun with a perturbed cut mesh
        {"name": "retry", "kind": "retry", "shape": "uv", "n": 64, "m": 8},
        # the registry's first consumer: cut-path edges of an 82k-triangle pair
        {"name": "cutpath", "kind": "cutpath", "shape": "ico", "n": 6, "m": 6},
        # MCUT's own calls when its front end runs here: 20k-triangle meshes
        {"name": "seam", "kind": "seam", "shape": "ico", "n": 5, "m": 5},
        # batches of independent pairs: many small ones ...
        {"name": "batch_small", "kind": "batch", "shape": "mix", "n": 16, "m": 8, "count": 96},
        # ... and the uneven mix (200-200k and 12-12k triangles a mesh)
        {"name": "batch_mix", "kind": "batch", "shape": "mix", "n": 100, "m": 32, "count": 320},
        # fragments on demand: a resident 165,620-triangle source and a burst of
        # crack sheets of 2k-50k triangles, registries kept
        {"name": "serve_burst", "kind": "serve", "shape": "sheets", "n": 91, "m": 158, "count": 12},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["device", "device", "device", "terrain", "host", "host", "retry", "cutpath", "seam", "batch", "batch",
                       "serve"])
    if kind == "device":
        if rng.random() < 0.3:
            return {"kind": "device", "shape": "uv", "n": _log(rng, 8, 400), "m": _log(rng, 1, 60)}
        return {"kind": "device", "shape": "grid", "n": _log(rng, 8, 250), "m": _log(rng, 8, 250)}
    if kind == "terrain":
        return {"kind": "device", "shape": "terrain", "n": _log(rng, 60, 1000), "m": _log(rng, 8, 64)}
    if kind == "host":
        if rng.random() < 0.5:
            return {"kind": "host", "shape": "polygon", "n": _log(rng, 2, 120), "m": _log(rng, 5, 48), "count": rng.randint(1, 4)}
        return {"kind": "host", "shape": "mix", "n": _log(rng, 8, 100), "m": _log(rng, 2, 32), "count": rng.randint(1, 16)}
    if kind == "retry":
        return {"kind": "retry", "shape": "uv", "n": 4 * _log(rng, 4, 60), "m": 2 * _log(rng, 1, 20)}
    if kind in ("cutpath", "seam"):
        return {"kind": kind, "shape": "grid", "n": _log(rng, 8, 80), "m": _log(rng, 8, 80)}
    if kind == "batch":
        n = _log(rng, 6, 100)
        return {"kind": "batch", "shape": "mix", "n": n, "m": _log(rng, 2, 32), "count": _log(rng, 2, 600 if n <= 20 else 200)}
    return {"kind": "serve", "shape": "sheets", "n": _log(rng, 20, 91), "m": _log(rng, 32, 158), "count": rng.randint(1, 12)}


# ---------------------------------------------------------------------------
# meshes: connectivity from the case, coordinates from the seed
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _ico(level):
    V, F, _ = mg.icosphere(level)
    return V, F


@functools.lru_cache(maxsize=128)
def _grid_sphere(n):
    V, F, _ = mg.geodesic_sphere(n)
    return V, F


@functools.lru_cache(maxsize=64)
def _uv(n):
    V, F, _ = mg.uv_sphere(n, max(3, n // 2), 1.0)
    return V, F


@functools.lru_cache(maxsize=64)
def _box(m, quads):
    V, F, S = mg.tessellated_box((0.0, 0.0, 0.0), 1.0, m, triangulate=not quads)
    return V, F, S


def _rotation(g):
    return mg.rotation_from_uniforms(*g.random(3))


def _noisy(g, V, amp=0.02):
    return V * (1.0 + amp * (2.0 * g.random(V.shape[0])[:, None] - 1.0))


def _prism(n, r, h, g):
    a = 2 * np.pi * np.arange(n) / n
    ring = np.stack([r * np.cos(a), r * np.sin(a), np.full(n, -h / 2)], 1)
    V = np.vstack([ring, ring + [0, 0, h]])
    i = np.arange(n)
    j = (i + 1) % n
    quads = np.stack([i, j, n + j, n + i], 1)
    F = np.concatenate([i[::-1], n + i, quads.ravel()])
    return V @ _rotation(g).T, F.astype(_U32), np.array([n, n] + [4] * n, _U32)


def _mix_pair(g, n, m):
    """A sphere of up to 20 n^2 triangles and a rotated box of up to 12 m^2
    that overlaps it by 10-60% of its radius, both sizes log-uniform."""
    fn = max(4, int(round(math.exp(math.log(4) + g.random() * (math.log(max(n, 4)) - math.log(4))))))
    bm = max(1, int(round(math.exp(g.random() * math.log(max(m, 1))))))
    V, F = _grid_sphere(fn)
    B, Fb, _ = _box(bm, False)
    s = 0.5 + g.random()
    d = g.standard_normal(3)
    d /= np.linalg.norm(d)
    C = (B * s) @ _rotation(g).T + d * (1.0 + s / 2 - (0.1 + 0.5 * g.random()))
    return (_noisy(g, V), F, None), (C, Fb, None)


def _terrain(g, cells, quads):
    """Fractal heights on a cells x cells grid of unit cells, on a 2^-12 grid,
    cut by a plane at a height that many of its vertices have."""
    h = torch.zeros(1, 1, cells + 1, cells + 1, dtype=torch.float64)
    for o in range(6):
        k = min(4 << o, cells)
        lat = torch.from_numpy(g.random((1, 1, k + 1, k + 1)))
        h += 0.5 ** o * torch.nn.functional.interpolate(lat, size=(cells + 1, cells + 1), mode="bilinear", align_corners=True)
    h = h.numpy().ravel()
    h = np.round((h - h.min()) / (h.max() - h.min()) * 0.2 * 4096.0) / 4096.0
    x, y = np.divmod(np.arange(h.size), cells + 1)
    V = np.stack([x, y, h], 1).astype(np.float64)
    i, j = np.divmod(np.arange(cells * cells), cells)
    a = i * (cells + 1) + j
    b = a + cells + 1
    F = np.stack([a, b, b + 1, a, b + 1, a + 1], 1).ravel()
    P, Fc, _ = mg.grid_patch(quads, 1.01 * cells)
    return (V, F.astype(_U32), None), (P + np.array([0.5 * cells, 0.5 * cells, 410.0 / 4096.0]), Fc, None)


def _sheet(g, most, side=3.0):
    """An open crack sheet of 2 q^2 triangles, q log-uniform up to `most`."""
    q = max(2, int(round(math.exp(math.log(max(2, most / 5)) + g.random() * math.log(max(1.0, most / max(2, most / 5)))))))
    G, F, _ = mg.grid_patch(q, side)
    h = 0.03 * np.sin(7.0 * G[:, 0] + 6.0 * g.random()) * np.cos(5.0 * G[:, 1] + 6.0 * g.random()) + 0.004 * g.random(G.shape[0])
    W = np.stack([G[:, 0], G[:, 1], h + 1.2 * g.random() - 0.6], 1)
    return W @ _rotation(g).T, F, None


def _meshes(case, seed):
    """The (source, cut) pairs of a case, from the seed alone."""
    g = np.random.Generator(np.random.PCG64(1000003 * int(seed) + 17))
    n, m, shape = case["n"], case["m"], case["shape"]
    if shape in ("ico", "grid"):
        make = _ico if shape == "ico" else _grid_sphere
        A, Fa = make(n)
        B, Fb = make(m)
        B = _noisy(g, B) @ _rotation(g).T
        B[:, 0] += 0.5
        return [((_noisy(g, A), Fa, None), (B, Fb, None))]
    if shape == "uv":
        A, Fa = _uv(n)
        B, Fb, _ = _box(m, False)
        if case["kind"] == "retry":  # the cube's face x = 1 touches the sphere's equator vertices
            s = 1.0 + np.round(g.random() * 64) / 256
            return [((A, Fa, None), (B * s + np.array([1.0 - s / 2, 0.25 * g.random(), 0.25 * g.random()]), Fb, None))]
        B = (B * 1.2) @ _rotation(g).T + np.array([0.4, 0.3, 0.2]) + 0.1 * g.random(3)
        return [((_noisy(g, A, 0.002), Fa, None), (B, Fb, None))]
    if shape == "terrain":
        return [_terrain(g, n, m)]
    if shape == "polygon":
        out = []
        for _ in range(case["count"]):
            A, Fa, Sa = _box(n, True)
            out.append(((A @ _rotation(g).T, Fa, Sa), _prism(m, 0.2 + 0.2 * g.random(), 0.8 + 0.4 * g.random(), g)))
        return out
    if shape == "mix":
        return [_mix_pair(g, n, m) for _ in range(case["count"])]
    if shape == "sheets":
        A, Fa = _grid_sphere(n)
        src = (_noisy(np.random.Generator(np.random.PCG64(6)), A), Fa, None)  # the resident mesh is the server's
        return [(src, _sheet(g, m)) for _ in range(case["count"])]
    raise ValueError(shape)


# ---------------------------------------------------------------------------
# the program: its handle, its inputs, its calls
# ---------------------------------------------------------------------------

_kept = {}


def _handle(case, make):
    """The context or server of the program that this case stands for."""
    key = tuple(sorted(case.items(), key=str))
    if key not in _kept:
        for h in _kept.values():
            h.close()
        _kept.clear()
        _kept[key] = make()
    return _kept[key]


def _up(a):
    """An array in GPU memory."""
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32) if a.dtype == _U32 else np.ascontiguousarray(a)).cuda()


def _resident(mesh):
    V, F, S = mesh
    t = [_up(V), _up(F), None if S is None else _up(S)]
    nf = F.size // 3 if S is None else S.size
    return t, fe.device_mesh(t[0].data_ptr(), t[1].data_ptr(), None if S is None else t[2].data_ptr(), V.shape[0], nf)


class _OnDevice:
    """An array of the library's in GPU memory, without a copy."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 3}


def _registry_on_device(ctx, count):
    """(edges, faces, points) of the last dispatch, where they lie."""
    C = fe.C
    e, f, p, k = C.c_void_p(), C.c_void_p(), C.c_void_p(), C.c_uint64()
    r = fe.lib().mcgpu_registry_device(ctx.h, C.byref(e), C.byref(f), C.byref(p), C.byref(k))
    if r != 0:
        raise fe.McgpuError(r, "mcgpu_registry_device")
    n = int(k.value)
    if n != count:
        raise RuntimeError("the registry has another length than the dispatch reported")
    if n == 0:
        return None
    return (torch.as_tensor(_OnDevice(e.value, (n,), "<i4"), device="cuda"),
            torch.as_tensor(_OnDevice(f.value, (n,), "<i4"), device="cuda"),
            torch.as_tensor(_OnDevice(p.value, (n, 3), "<f8"), device="cuda"))


def _move(seed):
    """The perturbation of a retry, within the widening of the cut boxes."""
    return (2.0 * np.random.Generator(np.random.PCG64(int(seed) + 5)).random(3) - 1.0) * 1e-4


# A registry's length depends on the meshes, and the context's next dispatch
# overwrites it: the program takes it into arrays of its own, whose length
# follows from the case, zero past the registry's end.

def _capacity(case):
    one = case["kind"] == "host"
    return int(8 * _sizes(case)[3] / (case["count"] if one else 1)) + 4096


def _arrays(case, device):
    n = _capacity(case)
    if device:
        return {"edges": torch.zeros(n, dtype=torch.int32, device="cuda"), "faces": torch.zeros(n, dtype=torch.int32, device="cuda"),
                "points": torch.zeros(n, 3, dtype=torch.float64, device="cuda")}
    return {"edges": np.zeros(n, _U32), "faces": np.zeros(n, _U32), "points": np.zeros((n, 3))}


def _take(out, **values):
    """Values into the program's arrays (they fit, or this raises)."""
    for k, v in values.items():
        out[k][:len(v)] = v
    return out


def _take_device(out, ctx, count):
    got = _registry_on_device(ctx, count)
    if got is not None:
        n = got[0].shape[0]
        if n > out["edges"].shape[0]:
            raise RuntimeError("a registry of %d entries does not fit" % n)
        for k, v in zip(("edges", "faces", "points"), got):
            out[k][:n].copy_(v)
    return out


def _soup(src, cut):
    """What MCUT holds before its front end: both meshes in its shifted
    coordinates and their face boxes, the cut faces' widened."""
    com, t, eps = _shift(src[0], cut[0])
    out = []
    for (V, F, _), e in ((src, 0.0), (cut, eps)):
        W = (V - com) + t
        T = W[F.reshape(-1, 3).astype(np.int64)]
        out.append(((W, F, None), np.hstack([T.min(1) - e, T.max(1) + e])))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        pairs = _meshes(case, seed)
        src, cuts = pairs[0][0], [p[1] for p in pairs]
        most = case["m"]
        srv = _handle(case, lambda: fe.Server(src, (most + 1) ** 2, 2 * most * most, slots=4))
        return {"case": case, "srv": srv, "cuts": cuts, "arrival": np.zeros(len(cuts)), "out": _arrays(case, False)}
    ctx = _handle(case, lambda: fe.Context(0))
    pairs = _meshes(case, seed)
    st = {"case": case, "ctx": ctx}
    if kind == "host":
        st["pairs"] = pairs
        st["out"] = [_arrays(case, False) for _ in pairs]
    elif kind == "seam":
        (s, sb), (c, cb) = _soup(*pairs[0])
        st.update(src=s, cut=c, sbox=sb, cbox=cb, out=_arrays(case, False))
        st["out"]["pairs"] = np.zeros((4 * (len(sb) + len(cb)), 2), _U32)
    elif kind == "batch":
        P = fe.pack_batch(pairs)
        st["keep"], meshes = [], []
        for side in ("src", "cut"):
            t, mesh = _resident(P[side])
            st["keep"].append(t)
            meshes.append(mesh)
        st.update(n=P["num_pairs"], src=meshes[0], cut=meshes[1], offs=[P[k] for k in ("src_vo", "src_fo", "cut_vo", "cut_fo")],
                  out=_arrays(case, True))
    else:
        st["keep"], meshes = [], []
        for mesh in pairs[0]:
            t, d = _resident(mesh)
            st["keep"].append(t)
            meshes.append(d)
        st.update(src=meshes[0], cut=meshes[1], nv=pairs[0][0][0].shape[0] + pairs[0][1][0].shape[0], out=_arrays(case, True))
        if kind == "retry":
            st["move"] = _move(seed)
        if kind == "cutpath":
            k = 2 * _capacity(case)
            st["out"].update({"src": np.zeros(k, _U32), "tgt": np.zeros(k, _U32), "groups": np.zeros(k, _U32),
                              "kinds": np.zeros(k, np.uint8), "cutfaces": np.zeros((k, 2), _U32)})
    torch.cuda.synchronize()
    return st


def _one(R, out):
    e, g, p = R.registry()
    return {"status": R.status, "count": len(e), **_take(out, edges=e, faces=g, points=p)}


def run(st):
    kind = st["case"]["kind"]
    if kind == "serve":
        srv = st["srv"]
        r = srv.run(st["cuts"], st["arrival"], keep_registries=True)
        got = [srv.registry(i, int(r["num_registry"][i])) for i in range(len(r))]
        e, g, p = (np.concatenate([x[k] for x in got]) for k in range(3))
        return {"status": r["status"], "registry": r["num_registry"].astype(np.int64),
                "candidates": r["num_candidate_pairs"].astype(np.int64), **_take(st["out"], edges=e, faces=g, points=p)}
    ctx = st["ctx"]
    if kind == "host":
        got = [_one(ctx.dispatch(*pair), out) for pair, out in zip(st["pairs"], st["out"])]
        return {"status": np.array([g["status"] for g in got]), "counts": np.array([g["count"] for g in got]),
                "registries": [{k: g[k] for k in ("edges", "faces", "points")} for g in got]}
    if kind == "seam":
        pairs = ctx.broad_phase(st["sbox"], st["cbox"])
        return _one(ctx.dispatch_narrow(st["src"], st["cut"], st["sbox"], st["cbox"], pairs), _take(st["out"], pairs=pairs))
    if kind == "batch":
        B = ctx.dispatch_batch_device(st["n"], st["src"], st["cut"], st["offs"])
        return {"status": B.status, "offsets": B.reg_offsets.astype(np.int64), **_take_device(st["out"], ctx, B.info.num_registry)}
    if kind == "retry":
        R = ctx.dispatch_device(st["src"], st["cut"], flags=fe.ENFORCE_GENERAL_POSITION)
        first = R.status
        if R.status_name == "GENERAL_POSITION_VIOLATION":
            R = ctx.redispatch_perturbed(st["move"], 0, st["nv"])
        return {"first": first, "status": R.status, **_take_device(st["out"], ctx, R.info.num_registry)}
    R = ctx.dispatch_device(st["src"], st["cut"])
    out = {"status": R.status, "candidates": R.counts["pairs"], "tests": R.counts["tests"],
           **_take_device(st["out"], ctx, R.info.num_registry)}
    if kind == "cutpath":
        P = R.cutpath()
        _take(out, cutfaces=P["faces"], **{k: P[k] for k in ("src", "tgt", "groups", "kinds")})
        out["short_group"] = P["short_group"]
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _sizes(case):
    """(vertices, faces, corners) of all meshes of a pass, on average over
    seeds, and the registry entries to expect."""
    n, m, shape = case["n"], case["m"], case["shape"]

    def sphere(k):
        return 10 * k * k + 2, 20 * k * k

    def box(k):
        return 6 * k * k + 2, 12 * k * k

    def mean_sq(a, b):  # mean of x^2, x log-uniform on [a, b]
        return a * a if b <= a else (b * b - a * a) / (2 * math.log(b / a))

    if shape in ("ico", "grid"):
        a, b = (sphere(2 ** n), sphere(2 ** m)) if shape == "ico" else (sphere(n), sphere(m))
        V, F = a[0] + b[0], a[1] + b[1]
        return V, F, 3 * F, 25 * math.sqrt(max(a[1], b[1]))
    if shape == "uv":
        k = max(3, n // 2)
        V, F = n * (k - 1) + 2, 2 * n * (k - 1)
        b = box(m)
        return V + b[0], F + b[1], 3 * (F + b[1]), 4 * (n + m)
    if shape == "terrain":
        V, F = (n + 1) ** 2 + (m + 1) ** 2, 2 * n * n + 2 * m * m
        return V, F, 3 * F, 4 * n
    if shape == "polygon":
        V, F = 6 * n * n + 2 + 2 * m, 6 * n * n + m + 2
        return V * case["count"], F * case["count"], (24 * n * n + 6 * m) * case["count"], 8 * n * case["count"]
    if shape == "mix":
        k = case["count"]
        a, b = mean_sq(4, max(n, 4)), mean_sq(1, max(m, 1))
        V, F = k * (10 * a + 6 * b + 4), k * (20 * a + 12 * b)
        return V, F, 3 * F, k * 12 * math.sqrt(a)
    k = case["count"]
    q = mean_sq(max(2, m / 5), m)
    return k * q, k * 2 * q, k * 6 * q, k * 8 * math.sqrt(q)  # the resident source is not read anew


def work(case):
    V, F, K, I = _sizes(case)
    faces = 4 * F if case["shape"] == "polygon" else 0
    extra = 96 * F if case["kind"] == "seam" else 0
    # coordinates and face lists read once, registry written; sums, shift and
    # boxes of every vertex and face, six orientation products an entry
    return {"bytes": float(24 * V + 4 * K + faces + extra + 32 * I), "flops": float(9 * V + 6 * K + 200 * I)}


# ---------------------------------------------------------------------------
# the same points in plain numpy
# ---------------------------------------------------------------------------

def _shift(Va, Vb):
    """Centre, translation and cut-box enlargement of a pair."""
    com = (np.cumsum(Va, axis=0)[-1] / len(Va) + np.cumsum(Vb, axis=0)[-1] / len(Vb)) / 2.0
    low = np.minimum(Va.min(0), Vb.min(0))
    d = com - low
    t = d + d / math.sqrt(float(d @ d))
    ext = (Vb.max(0) + t) - (Vb.min(0) + t)
    return com, t, math.sqrt(float(ext @ ext)) * 1e-4


def _padded(F, S):
    """Faces as rows of vertex ids, -1 past a face's last corner."""
    if S is None:
        return F.reshape(-1, 3).astype(np.int64)
    S = S.astype(np.int64)
    out = np.full((S.size, int(S.max())), -1, np.int64)
    out[np.arange(out.shape[1])[None] < S[:, None]] = F
    return out


def _edges(P, first):
    """Edges in order of first use, with the direction of that use; a face's
    list starts at its corner `first`."""
    n = (P >= 0).sum(1)
    col = np.arange(P.shape[1])[None]
    ok = col < n[:, None]
    a = np.take_along_axis(P, (col + first) % n[:, None], 1)
    b = np.take_along_axis(P, (col + first + 1) % n[:, None], 1)
    a, b = a[ok], b[ok]
    _, i = np.unique(np.minimum(a, b) * (P.max() + 1) + np.maximum(a, b), return_index=True)
    i.sort()
    return a[i], b[i]


def _cells(lo, hi, org, size, dims):
    """(item, cell) of every grid cell a box touches."""
    a = np.clip(((lo - org) / size).astype(np.int64), 0, dims - 1)
    b = np.clip(((hi - org) / size).astype(np.int64), 0, dims - 1)
    n = b - a + 1
    k = n.prod(1)
    item = np.repeat(np.arange(len(lo)), k)
    r = np.arange(k.sum()) - np.repeat(np.cumsum(k) - k, k)
    n, a = n[item], a[item]
    z = r % n[:, 2]
    y = (r // n[:, 2]) % n[:, 1]
    x = r // (n[:, 2] * n[:, 1])
    return item, ((a[:, 0] + x) * dims[1] + a[:, 1] + y) * dims[2] + a[:, 2] + z


def _near(lo0, hi0, lo1, hi1):
    """Pairs of boxes that overlap."""
    org, top = np.maximum(lo0.min(0), lo1.min(0)), np.minimum(hi0.max(0), hi1.max(0))
    A = np.nonzero((lo0 <= top).all(1) & (hi0 >= org).all(1))[0]
    B = np.nonzero((lo1 <= top).all(1) & (hi1 >= org).all(1))[0]
    if not len(A) or not len(B):
        return A[:0], B[:0]
    lo0, hi0, lo1, hi1 = lo0[A], hi0[A], lo1[B], hi1[B]
    size = 1.5 * max((hi0 - lo0).mean(), (hi1 - lo1).mean()) + 1e-12
    dims = np.clip(np.ceil((top - org) / size).astype(np.int64), 1, 512)
    size = np.maximum((top - org) / dims, 1e-300)
    i, ci = _cells(lo0, hi0, org, size, dims)
    j, cj = _cells(lo1, hi1, org, size, dims)
    o = np.argsort(cj, kind="stable")
    j, cj = j[o], cj[o]
    s, e = np.searchsorted(cj, ci, "left"), np.searchsorted(cj, ci, "right")
    k = e - s
    I = np.repeat(i, k)
    J = j[np.repeat(s, k) + np.arange(k.sum()) - np.repeat(np.cumsum(k) - k, k)]
    ok = ((lo0[I] <= hi1[J]) & (hi0[I] >= lo1[J])).all(1)
    u = np.unique(I[ok] * len(B) + J[ok])
    return A[u // len(B)], B[u % len(B)]


def _crossings(W, ea, eb, P):
    """Rows (edge, face, point) where a segment of vertices W crosses a face
    of P (rows of vertex ids of W)."""
    n = (P >= 0).sum(1)
    nxt = np.take_along_axis(P, (np.arange(P.shape[1])[None] + 1) % n[:, None], 1)
    ok = P >= 0
    X, Y = W[np.where(ok, P, P[:, :1])], W[np.where(ok, nxt, P[:, :1])]
    use = ok[:, :, None]
    nrm = np.stack([((X[..., i] - Y[..., i]) * (X[..., j] + Y[..., j]) * ok).sum(1) for i, j in ((1, 2), (2, 0), (0, 1))], 1)
    nrm /= np.maximum(np.linalg.norm(nrm, axis=1), 1e-300)[:, None]
    d = (nrm * (X * use).sum(1)).sum(1) / n
    ends = W[ea], W[eb]
    E, G = _near(np.minimum(*ends), np.maximum(*ends), X.min(1), X.max(1))
    q, r, nn = W[ea[E]], W[eb[E]], nrm[G]
    dq, dr = (q * nn).sum(1) - d[G], (r * nn).sum(1) - d[G]
    c = dq * dr < 0
    E, G, q, r, nn, dq, dr = E[c], G[c], q[c], r[c], nn[c], dq[c], dr[c]
    p = q + (dq / (dq - dr))[:, None] * (r - q)
    drop = np.abs(nn).argmax(1)
    ax = np.array([[1, 2], [0, 2], [0, 1]])[drop]
    take = lambda a: np.take_along_axis(a, ax.reshape(ax.shape[:1] + (1,) * (a.ndim - 2) + (2,)), -1)  # noqa: E731
    x, y, z = take(X[G]), take(Y[G]), take(p)[:, None, :]
    span = (x[..., 1] > z[..., 1]) != (y[..., 1] > z[..., 1])
    dy = np.where(span, y[..., 1] - x[..., 1], 1.0)
    inside = ((span & ok[G] & (z[..., 0] < (y[..., 0] - x[..., 0]) * (z[..., 1] - x[..., 1]) / dy + x[..., 0])).sum(1) % 2) == 1
    return E[inside], G[inside], p[inside]


def _points(src, cut, move=None, shifted=False):
    """Registry points of one pair in general position, sorted by (edge, face)."""
    com, t, _ = _shift(src[0], cut[0])
    A, B = ((src[0], cut[0]) if shifted else ((src[0] - com) + t, (cut[0] - com) + t))
    W = np.vstack([A, B if move is None else B + move])
    Ps, Pc = _padded(src[1], src[2]), _padded(cut[1], cut[2])
    a0, b0 = _edges(Ps, 0)
    a1, b1 = _edges(Pc, 1)
    nv, nf = len(src[0]), len(Ps)
    Pc = np.where(Pc >= 0, Pc + nv, -1)
    E0, G0, p0 = _crossings(W, a0, b0, Pc)
    E1, G1, p1 = _crossings(W, a1 + nv, b1 + nv, Ps)
    o = np.lexsort((np.concatenate([G0 + nf, G1]), np.concatenate([E0, E1 + len(a0)])))
    return np.concatenate([p0, p1])[o]


def exact(case, seed):
    kind = case["kind"]
    if case["shape"] == "terrain":  # not in general position: no such points
        return None
    if _sizes(case)[1] + (case["count"] * 20 * case["n"] ** 2 if kind == "serve" else 0) > 2_500_000:
        return None  # half a minute in numpy
    pairs = _meshes(case, seed)

    def whole(p):
        out = np.zeros((_capacity(case), 3))
        out[:len(p)] = p
        return {"points": out}

    if kind == "seam":
        (s, _), (c, _) = _soup(*pairs[0])
        return whole(_points(s, c, shifted=True))
    if kind == "host":
        return {"registries": [whole(_points(*p)) for p in pairs]}
    move = _move(seed) if kind == "retry" else None
    return whole(np.concatenate([_points(*p, move=move) for p in pairs]))
