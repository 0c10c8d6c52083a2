"""The work this framework is used for, as cases that can be timed.

A case is a dict of plain values; `prepare` makes what a user's program holds
before the call (meshes with their hierarchies, packed queries, device
buffers, scorers), `run` is one pass through the public entry points of
`c2a_amd`, and `work` says what such a pass cannot do without.

Sizes are the repository's own: the (2,3) torus-knot tubes (1,024 to 8,192
triangles), the uneven mesh table (80 to 81,920 triangles), the bunny of the
reference's demo (69,664 triangles) and the noisy UV spheres (up to 262,144
triangles); batches from one query to 16,384.
"""
import functools
import math

import numpy as np
import torch

import c2a_amd as G
from c2a_amd import learn
from c2a_amd import workloads as W


def listed():
    return [
        # A program that solves one query at a time, as the reference's own
        # loop does (C2A_Solve: time of contact, then the contacts there).
        {"name": "solve_one", "kind": "solve", "nq": 1, "seg": 256, "ring": 16, "contacts": 1,
         "strict": 0},
        # A serving loop: a few queries on small meshes, device buffers owned
        # by the caller, nothing allocated per call.
        {"name": "serve_64", "kind": "serve", "nq": 64, "seg": 64, "ring": 8, "strict": 0},
        # The reference's demo: 303 frames of two bunnies, with contacts.
        {"name": "demo_303", "kind": "batch", "shape": "bunny", "nq": 303, "order": "plain",
         "contacts": 1, "strict": 0},
        # The headline batch: two knots, 4096 independent motions.
        {"name": "knot_4096", "kind": "batch", "shape": "knot", "seg": 256, "ring": 16,
         "nq": 4096, "order": "plain", "contacts": 0, "strict": 0},
        # Many meshes of very different sizes in one batch (a scene).
        {"name": "uneven_8191", "kind": "batch", "shape": "uneven", "nq": 8191,
         "order": "plain", "contacts": 0, "strict": 0},
        # The largest meshes, passing each other almost in touch.
        {"name": "grazing_256", "kind": "batch", "shape": "sphere", "lon": 512, "lat": 256,
         "nq": 256, "order": "plain", "contacts": 0, "strict": 0},
        # The learned sibling order with the shipped scorer.
        {"name": "learned_2048", "kind": "batch", "shape": "knot", "seg": 256, "ring": 16,
         "nq": 2048, "order": "learned", "contacts": 0, "strict": 0},
        # Static proximity: exact distance, contact pairs, tolerance.
        {"name": "distance_16384", "kind": "distance", "nq": 16384, "seg": 256, "ring": 16,
         "qsize": 2, "rel": 0.0},
        {"name": "collide_2048", "kind": "collide", "nq": 2048, "seg": 256, "ring": 16,
         "flag": 1, "cap": 256},
        {"name": "tolerance_4096", "kind": "tolerance", "nq": 4096, "seg": 256, "ring": 16,
         "tol": 0.05, "qsize": 2},
        # A deforming body: its hierarchy built on the GPU, refitted to the
        # moved triangles, then a few distances against itself.
        {"name": "deform_262144", "kind": "deform", "lon": 512, "lat": 256, "nq": 64},
        # Training of the pair scorer (forward, backward, Adam).
        {"name": "train_65536", "kind": "train", "n": 65536, "epochs": 2, "batch": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "serve", "knot", "uneven", "sphere", "distance", "collide",
                       "tolerance", "deform", "train"])
    ring = rng.randint(8, 16)
    seg = _log(rng, 64, 4096 // ring)
    if kind == "solve":
        return {"kind": "solve", "nq": _log(rng, 1, 32), "seg": seg, "ring": ring,
                "contacts": rng.randint(0, 1), "strict": rng.randint(0, 1)}
    if kind == "serve":
        return {"kind": "serve", "nq": _log(rng, 16, 1024), "seg": seg, "ring": ring,
                "strict": rng.randint(0, 1)}
    if kind == "knot":
        return {"kind": "batch", "shape": "knot", "seg": seg, "ring": ring,
                "nq": _log(rng, 64, 4096), "order": rng.choice(["plain", "plain", "learned"]),
                "contacts": rng.randint(0, 1), "strict": rng.randint(0, 1)}
    if kind == "uneven":
        return {"kind": "batch", "shape": "uneven", "nq": _log(rng, 256, 8191),
                "order": rng.choice(["plain", "plain", "learned"]), "contacts": 0,
                "strict": rng.randint(0, 1)}
    if kind == "sphere":
        lat = _log(rng, 64, 256)
        return {"kind": "batch", "shape": "sphere", "lon": 2 * lat - rng.randint(0, 15),
                "lat": lat, "nq": _log(rng, 32, 192), "order": "plain", "contacts": 0,
                "strict": rng.randint(0, 1)}
    if kind == "distance":
        return {"kind": "distance", "nq": _log(rng, 256, 16384), "seg": seg, "ring": ring,
                "qsize": rng.choice([2, 2, 16]), "rel": rng.choice([0.0, 0.0, 0.05])}
    if kind == "collide":
        return {"kind": "collide", "nq": _log(rng, 64, 2048), "seg": seg, "ring": ring,
                "flag": rng.randint(1, 2), "cap": _log(rng, 16, 256)}
    if kind == "tolerance":
        return {"kind": "tolerance", "nq": _log(rng, 256, 4096), "seg": seg, "ring": ring,
                "tol": round(math.exp(rng.uniform(math.log(0.005), math.log(0.2))), 4),
                "qsize": rng.choice([2, 2, 16])}
    if kind == "deform":
        lat = _log(rng, 24, 240)
        return {"kind": "deform", "lon": 2 * lat + rng.randint(1, 15), "lat": lat,
                "nq": _log(rng, 1, 64)}
    return {"kind": "train", "n": _log(rng, 3000, 65536), "epochs": rng.randint(1, 2),
            "batch": _log(rng, 500, 4096)}


# ---------------------------------------------------------------------------
# geometry (the same for every seed) and inputs (made from the seed)
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _knot(seg, ring):
    t, idx = W.torus_knot(n_seg=seg, n_ring=ring)
    return t.reshape(-1, 9), idx


@functools.lru_cache(maxsize=None)
def _sphere(lon, lat):
    t, idx = W.uv_sphere(lon, lat, 0.1, 3)
    return t.reshape(-1, 9), idx


@functools.lru_cache(maxsize=None)
def _uneven():
    return W.uneven_meshes()


@functools.lru_cache(maxsize=None)
def _bunny():
    t, idx = W.bunny()
    return t, idx, W.demo_queries()


def _knots(case):
    t, idx = _knot(case["seg"], case["ring"])
    return [G.Mesh(t, vidx=idx), G.Mesh(t, vidx=idx)]


def _batch_inputs(case, seed):
    """(meshes, poses, mesh pairs, tolerances) of a batch."""
    nq, shape = case["nq"], case["shape"]
    if shape == "knot":
        return _knots(case), W.knot_queries(nq, seed, 0.3), None, (1e-3, 1e-4)
    if shape == "uneven":
        tab = _uneven()
        meshes = [G.Mesh(t, vidx=i, device=True) for t, i, _ in tab]
        *P, mp = W.uneven_queries(nq, seed, [len(t) for t, _, _ in tab], [r for _, _, r in tab])
        return meshes, P, mp, (1e-3, 1e-4)
    if shape == "bunny":
        # the demo's frames, object 2's path moved by up to 2% of its span
        t, idx, P = _bunny()
        P = [p[:nq].copy() for p in P]
        span = float(np.abs(t.reshape(-1, 3)).max())
        off = W.Rng(seed, 21).uniform(3 * len(P[0]), -0.02, 0.02).reshape(-1, 3) * span
        P[2][:, 9:] += off
        P[3][:, 9:] += off
        mesh = G.Mesh(t, vidx=idx, device=True)
        return [mesh, mesh], P, None, (1e-4, 1e-4)
    t, idx = _sphere(case["lon"], case["lat"])
    mesh = G.Mesh(t, vidx=idx, device=True)
    return [mesh, mesh], W.grazing_queries(nq, seed), None, (1e-3, 1e-4)


def _static_inputs(case, seed):
    """Knots at the start poses of the knot workload's motions."""
    P = W.knot_queries(case["nq"], seed, 0.3)
    poses = np.ascontiguousarray(np.concatenate([P[0], P[2]], axis=1))
    return poses, np.tile(np.array([0, 1], np.int32), (case["nq"], 1))


def _samples(case, seed):
    """Feature rows and labels with the ranges the traversal's samples have:
    lengths over the body's radius, a rotation, logs down to log(1e-4)."""
    r = np.random.default_rng(seed)
    n = case["n"]
    X = np.zeros((n, G.NF), np.float32)
    X[:, 0:6] = np.exp(r.uniform(math.log(1e-3), 0.0, (n, 6)))
    X[:, 6:9] = r.normal(0.0, 0.5, (n, 3))
    X[:, 9:18] = W.quat_to_matrix(r.normal(size=(n, 4))).reshape(n, 9)
    X[:, 18:22] = np.log(np.exp(r.uniform(-9.2, 0.7, (n, 4))) + 1e-4)
    X[:, 22:24] = r.integers(1, 18, (n, 2)) * 0.0625
    X[:, 24:26] = r.uniform(0.2, 1.0, (n, 2))
    X[:, 26:30] = r.uniform(0.1, 3.0, (n, 4))
    X[:, 30] = r.uniform(0.2, 1.0, n)
    X[:, 31] = r.integers(0, 3, n) / 3.0
    y = 0.8 * X[:, 18] + 0.3 * np.log(X[:, 4] + X[:, 5] + 1e-3) + r.normal(0.0, 0.3, n)
    return X, np.maximum(y, math.log(1e-4)).astype(np.float32)


def _weights(seed):
    """He-uniform weights and zero biases, as a new scorer starts."""
    r = np.random.default_rng(seed + 1)
    w1 = r.uniform(-1, 1, (32, 64)) * math.sqrt(6 / 32)
    w2 = r.uniform(-1, 1, (64, 64)) * math.sqrt(6 / 64)
    w3 = r.uniform(-1, 1, 64) * math.sqrt(6 / 64) * 0.5
    z = np.zeros(64)
    return np.concatenate([w1.ravel(), z, w2.ravel(), z, w3, [0.0]]).astype(np.float32)


LR = 2e-3
_RESULT_F64 = list(range(0, 21)) + list(range(26, 41))   # words of c2a_result


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        # the reference's loop builds its two models once, then solves per frame
        meshes = _knots(case)
        P = W.knot_queries(case["nq"], seed, 1.0)
        params = G.default_params(tol_d=1e-3, with_contacts=case["contacts"],
                                  strict=case["strict"])
        return {"kind": kind, "meshes": meshes, "queries": G.make_queries(*P), "params": params}
    if kind == "serve":
        meshes = _knots(case)
        P = W.knot_queries(case["nq"], seed, 0.3)
        params = G.default_params(tol_d=1e-3, with_contacts=0, strict=case["strict"])
        # the first launch puts the meshes on the device
        G.ccd_batch(meshes, G.make_queries(*[p[:1] for p in P]), params)
        nq = case["nq"]
        motions = torch.from_numpy(G.motion_records(*P)).cuda()
        pairs = torch.tensor([[0, 1]] * nq, dtype=torch.int32, device="cuda")
        out = torch.zeros((nq, G.RESULT_DTYPE.itemsize // 8), dtype=torch.float64, device="cuda")
        return {"kind": kind, "meshes": meshes, "motions": motions, "pairs": pairs, "out": out,
                "nq": nq, "params": params}
    if kind == "batch":
        meshes, P, mp, (tol_d, tol_t) = _batch_inputs(case, seed)
        scorer = G.Scorer(path=learn.DEFAULT_SCORER) if case["order"] == "learned" else None
        kw = dict(order=G.ORDER_LEARNED, scorer=scorer) if scorer else {}
        params = G.default_params(tol_d=tol_d, tol_t=tol_t, with_contacts=case["contacts"],
                                  strict=case["strict"], **kw)
        return {"kind": kind, "batch": G.Batch(meshes, G.make_queries(*P, mesh_pairs=mp), params,
                                               scorer=scorer)}
    if kind in ("distance", "collide", "tolerance"):
        poses, pairs = _static_inputs(case, seed)
        return {"kind": kind, "meshes": _knots(case), "poses": poses, "pairs": pairs,
                "case": case}
    if kind == "deform":
        t, idx = _sphere(case["lon"], case["lat"])
        r = np.random.default_rng(seed)
        v = t.reshape(-1, 3)
        k, ph = r.normal(0.0, 3.0, (2, 3)), r.uniform(0, 2 * np.pi, 2)
        tris = [np.ascontiguousarray((v * (1 + 0.05 * np.sin(v @ k[i] + ph[i]))[:, None])
                                     .reshape(-1, 9)) for i in range(2)]
        rng = W.Rng(seed, 9)
        R1, R2 = (W.quat_to_matrix(W.random_quats(rng, case["nq"])) for _ in range(2))
        d = r.normal(size=(case["nq"], 3))
        T = d / np.linalg.norm(d, axis=1, keepdims=True) * r.uniform(2.0, 3.0, (case["nq"], 1))
        poses = np.concatenate([W.pack_poses(R1, 0 * T), W.pack_poses(R2, T)], axis=1)
        return {"kind": kind, "tris": tris, "idx": idx, "poses": poses,
                "pairs": np.zeros((case["nq"], 2), np.int32)}
    X, y = _samples(case, seed)
    return {"kind": kind, "scorer": G.Scorer(seed), "X": X, "y": y, "p0": _weights(seed),
            "case": case, "seed": seed & 0xffff}


def _fields(a, names):
    return {f: a[f] for f in names}


_CCD = ("toc", "distance", "mint", "R_toc", "T_toc", "p1", "p2", "bv_tests", "tri_tests",
        "numCA", "collisionfree", "num_contact", "last_tri", "flags", "R", "T", "abs_err",
        "rel_err", "UpboundTOC")
_DIST = ("distance", "p1", "p2", "bv_tests", "tri_tests", "last_tri", "flags")
_STATIC = ("distance", "p1", "p2", "bv_tests", "tri_tests", "tri", "found", "flags")


def run(s):
    kind = s["kind"]
    if kind == "solve":
        return _fields(G.ccd_batch(s["meshes"], s["queries"], s["params"]), _CCD)
    if kind == "serve":
        out = s["out"]
        G.ccd_batch_noalloc(s["meshes"], s["motions"].data_ptr(), s["pairs"].data_ptr(), None,
                            s["nq"], s["params"], out.data_ptr(),
                            stream=torch.cuda.current_stream().cuda_stream)
        return {"numbers": out[:, _RESULT_F64], "counts": out[:, 21:23].view(torch.int64),
                "ints": out.view(torch.int32)[:, 46:52]}
    if kind == "batch":
        s["batch"].run()
        return _fields(s["batch"].fetch(), _CCD)
    if kind == "distance":
        c = s["case"]
        if c["qsize"] > 2:
            r = G.distance_queue(s["meshes"], s["poses"], s["pairs"], c["qsize"],
                                 rel_err=c["rel"])
        else:
            r = G.distance(s["meshes"], s["poses"], s["pairs"], rel_err=c["rel"])
        return _fields(r, _DIST)
    if kind == "collide":
        c = s["case"]
        r, pairs = G.collide_pairs(s["meshes"], s["poses"], s["pairs"], flag=c["flag"],
                                   cap=c["cap"])
        # the pairs a query found; the rest of its list holds none
        pairs[np.arange(c["cap"]) >= r["found"][:, None]] = -1
        return dict(_fields(r, _STATIC), pairs=pairs)
    if kind == "tolerance":
        c = s["case"]
        return _fields(G.tolerance(s["meshes"], s["poses"], s["pairs"], c["tol"], c["qsize"]),
                       _STATIC)
    if kind == "deform":
        mesh = G.Mesh(s["tris"][0], vidx=s["idx"], device=True)
        order = mesh.tri_ids()
        mesh.refit(s["tris"][1])
        r = G.distance([mesh], s["poses"], s["pairs"])
        return dict(_fields(r, _DIST), order=order)
    c = s["case"]
    s["scorer"].set_params(s["p0"])
    losses = s["scorer"].train(s["X"], s["y"], epochs=c["epochs"], batch=c["batch"], lr=LR,
                               seed=s["seed"])
    return {"params": s["scorer"].params(), "losses": losses}


# Mean volume pairs tested per query (counted once at the listed sizes); a
# pair test is two node records and about 400 flops, a query two motions and
# a result record.
_PAIRS = {"knot": 25000, "uneven": 10300, "bunny": 23500, "sphere": 148000}


def work(case):
    kind = case["kind"]
    if kind == "train":
        rows = case["n"] * case["epochs"]
        return {"bytes": case["n"] * 33 * 4 + rows * 4 + 6 * 6337 * 4, "flops": rows * 3 * 2 * 6208}
    if kind == "deform":
        n = 2 * case["lon"] * case["lat"]
        levels = math.log2(n) + 1
        return {"bytes": n * (2 * 72 + 12 + 4) + case["nq"] * 300,
                "flops": 2 * n * levels * 150 + case["nq"] * 5000 * 400}
    if kind == "batch" and case["shape"] != "knot":
        ntri = {"uneven": 121000, "bunny": 69664}.get(case["shape"]) or 2 * case["lon"] * case["lat"]
        pairs = _PAIRS[case["shape"]]
        if case["shape"] == "sphere":
            pairs *= math.sqrt(ntri / 262144)
    else:
        ntri = 4 * case["seg"] * case["ring"]
        per = _PAIRS["knot"] if kind in ("solve", "serve", "batch") else 4600
        pairs = per * math.sqrt(ntri / 16384)
    return {"bytes": ntri * (2 * 256 + 72) + case["nq"] * 728,
            "flops": case["nq"] * pairs * 400}


# ---------------------------------------------------------------------------
# 64-bit values.  The traversals' outputs are decisions of a depth-first
# search (which pairs are visited, when it stops), which no direct formula
# gives; brute force over all triangle pairs takes minutes at these sizes.
# The scorer's training is plain arithmetic.
# ---------------------------------------------------------------------------
_M64 = (1 << 64) - 1


def _mix(z):
    z = (z + 0x9E3779B97F4A7C15) & _M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    return z ^ (z >> 31)


def exact(case, seed):
    if case["kind"] != "train":
        return None
    X, y = _samples(case, seed)
    n, nb = case["n"], case["batch"]
    X, y = (torch.from_numpy(a).double().cuda() for a in (X, y))
    p = torch.from_numpy(_weights(seed)).double().cuda()
    mom, vel, step, losses = torch.zeros_like(p), torch.zeros_like(p), 0, []
    st = _mix((seed & 0xffff) ^ 0xA11CE)
    for _ in range(case["epochs"]):
        perm = list(range(n))
        for i in range(n - 1, 0, -1):
            st = _mix(st)
            j = st % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        perm = torch.tensor(perm, device="cuda")
        total = torch.zeros((), dtype=torch.float64, device="cuda")
        for b in range(0, n, nb):
            rows = perm[b:b + nb]
            x, t = X[rows], y[rows]
            w1, b1 = p[:2048].view(32, 64), p[2048:2112]
            w2, b2, w3, b3 = p[2112:6208].view(64, 64), p[6208:6272], p[6272:6336], p[6336]
            h1 = (x @ w1 + b1).clamp(min=0)
            h2 = (h1 @ w2 + b2).clamp(min=0)
            e = h2 @ w3 + b3 - t
            total += (e * e).sum()
            dy = e * (2.0 / len(rows))
            d2 = (dy[:, None] * w3) * (h2 > 0)
            d1 = (d2 @ w2.t().contiguous()) * (h1 > 0)
            g = torch.cat([(x.t() @ d1).reshape(-1), d1.sum(0), (h1.t() @ d2).reshape(-1),
                           d2.sum(0), h2.t() @ dy, dy.sum()[None]])
            step += 1
            mom = 0.9 * mom + 0.1 * g
            vel = 0.999 * vel + 0.001 * g * g
            mh, vh = mom / (1 - 0.9 ** step), vel / (1 - 0.999 ** step)
            p = p - LR * mh / (vh.sqrt() + 1e-8)
        losses.append(total / n)
    return {"params": p, "losses": torch.stack(losses)}
