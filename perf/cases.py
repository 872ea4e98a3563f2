"""The work that a user has this engine do, as cases to time.

Every case goes through the public entry points (`voronoi_amd.native`, the
binding of the C ABI in include/vd_api.h):

  lloyd    one mesh resident in a context: the caller sets sites, runs Lloyd
           iterations and reads the sites back
  step     one iteration in its three steps, with the per-site volumes and
           first moments and the sites read back
  batch    many independent instances in one context, each iteration a replay
           of one captured graph
  serve    a set of jobs submitted to the job server and stepped until done
  program  the reference's whole-program driver on host buffers
  knn_dev  the reference's device kNN on pitched device arrays
  kn       the reference's grid kNN problem: prepare, solve, read the lists

Meshes and sites are the seeded constructions of the benchmark and the tests:
jittered unit cubes of 6 n^3 tets with uniform sites (a tenth of the tets, or
the benchmark's own counts) and the voxelised torus with sites from a Gaussian
mixture, in the [0,1000]^3 frame.  Neighbour and candidate counts are the
benchmark's (site_k 90, tet_k 64 or 96) or the defaults (site_k 90, tet_k from
the reference's heuristic, written as 0).
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "3d-voronoi-gpu_amd"))

from voronoi_amd import meshgen, native  # noqa: E402

FAST = {"form": "site", "accum": "f64", "moments": "robust"}


def _lloyd(kind, n, n_sites, iters, tk=64, k=90, mesh="cube", **cfg):
    return {"kind": kind, "mesh": mesh, "n": n, "n_sites": n_sites, "iters": iters, "tk": tk, "k": k, **FAST, **cfg}


def listed():
    return [
        # the smallest calls, where launches and host work count: a mesh of 1,296 tets
        # with an odd number of sites, as the tests use
        dict(_lloyd("lloyd", 6, 131, 10), name="lloyd_1k_tets"),
        # the smallest instance of the benchmark's batch, alone
        dict(_lloyd("lloyd", 12, 1037, 10), name="lloyd_10k_tets"),
        # the benchmark's small workload (48,000 tets, 2,000 sites, one iteration):
        # volumes and centroids of given sites, step by step
        dict(_lloyd("step", 20, 2000, 1), name="step_48k_tets"),
        # a mid-size mesh with the library's defaults (FP32 sums, the reference's
        # moments, tet_k from its heuristic), odd sizes
        dict(_lloyd("lloyd", 29, 14633, 5, tk=0, accum="f32", moments="reference"), name="lloyd_146k_tets_defaults"),
        # the benchmark's headline: 998,250 tets, 100,000 uniform sites, the chain of 10
        dict(_lloyd("lloyd", 55, 100000, 10), name="lloyd_1m_tets"),
        # the benchmark's non-uniform domain: torus of 820,272 tets, 200,000 sites of
        # 50x density contrast, tet_k 96
        dict(_lloyd("lloyd", 96, 200000, 2, tk=96, mesh="torus"), name="lloyd_torus_820k_tets"),
        # the cell -> tet formulation (the drop-in's default) on a mid-size mesh
        dict(_lloyd("lloyd", 40, 38400, 2, form="cells"), name="cells_384k_tets"),
        # the benchmark's batch workload with 32 of its 256 instances: 10k..547k tets each
        {"kind": "batch", "instances": 32, "lo": 12, "hi": 45, "iters": 3, "tk": 64, "k": 90, **FAST,
         "name": "batch_32_instances"},
        # the served workload's mix: 12 jobs of 5..20 iterations through the job server
        {"kind": "serve", "jobs": 12, "lo": 12, "hi": 30, "iters_lo": 5, "iters_hi": 20, "tk": 64, "k": 90, **FAST,
         "name": "serve_12_jobs"},
        # the reference's driver as its command line runs it: cells, FP32 sums, tet_k from
        # the heuristic, three iterations with their files, at the size of its example
        dict(_lloyd("program", 17, 3001, 3, tk=0, form="cells", accum="f32", moments="reference"),
             name="program_29k_tets"),
        # the reference's device kNN as its driver calls it: every tet's candidates
        {"kind": "knn_dev", "n_ref": 100000, "n_query": 998250, "k": 64, "name": "knn_dev_100k_x_1m"},
        # the reference's grid kNN at the size of its example
        {"kind": "kn", "n_ref": 3001, "n_query": 3001, "k": 90, "name": "kn_3k"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lloyd", "lloyd", "lloyd", "step", "cells", "torus", "batch", "serve", "program", "knn_dev", "kn"])
    opt = {"accum": rng.choice(["f64", "f64", "f32"]), "moments": rng.choice(["robust", "robust", "reference"])}
    if kind in ("lloyd", "step"):
        n = _log_int(rng, 6, 55)
        ns = max(120, int(6 * n ** 3 * rng.uniform(0.04, 0.12)))
        return _lloyd(kind, n, ns, 1 if kind == "step" else rng.randint(1, 8), tk=rng.choice([0, 32, 64, 64]), **opt)
    if kind == "cells":
        n = _log_int(rng, 8, 44)
        return _lloyd("lloyd", n, max(120, int(6 * n ** 3 * rng.uniform(0.05, 0.1))), rng.randint(1, 2), form="cells", **opt)
    if kind == "torus":
        n = _log_int(rng, 24, 96)
        ns = max(200, int(0.92 * n ** 3 * rng.uniform(0.05, 0.24)))
        return _lloyd("lloyd", n, ns, rng.randint(1, 2), tk=rng.choice([64, 96]), mesh="torus", **opt)
    if kind == "batch":
        return {"kind": "batch", "instances": _log_int(rng, 2, 32), "lo": 12, "hi": rng.randint(20, 40),
                "iters": rng.randint(2, 4), "tk": 64, "k": 90, **FAST}
    if kind == "serve":
        return {"kind": "serve", "jobs": rng.randint(2, 12), "lo": 12, "hi": rng.randint(14, 30), "iters_lo": 5,
                "iters_hi": rng.randint(6, 20), "tk": 64, "k": 90, **FAST}
    if kind == "program":
        n = _log_int(rng, 8, 24)
        return _lloyd("program", n, max(120, int(6 * n ** 3 * rng.uniform(0.05, 0.1))), rng.randint(1, 3), tk=0,
                      form="cells", accum="f32", moments="reference")
    if kind == "knn_dev":
        return {"kind": "knn_dev", "n_ref": _log_int(rng, 300, 100000), "n_query": _log_int(rng, 300, 998250),
                "k": rng.choice([8, 20, 50, 64, 90, 96])}
    n = _log_int(rng, 300, 100000)
    return {"kind": "kn", "n_ref": n, "n_query": n, "k": rng.choice([20, 64, 90])}


def _cfg(case):
    return {"site_k": case["k"], "tet_k": case["tk"], "form": case["form"], "accum": case["accum"],
            "moments": case["moments"]}


def _problem(case, seed):
    return meshgen.make_problem(case["mesh"], case["n"], case["n_sites"], seed=1000 + 17 * seed)


def _sizes(case, count):
    return [int(n) for n in meshgen.batch_sizes(count, case["lo"], case["hi"])]


def _instances(case, seed, count):
    return [meshgen.make_problem("cube", n, 6 * n ** 3 // 10, seed=100000 + 977 * seed + i)
            for i, n in enumerate(_sizes(case, count))]


def _uniform(seed, n):
    return (1000.0 * meshgen.uniform_sites(n, seed=500 + seed).astype(np.float64)).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("lloyd", "step"):
        verts, tets, s["sites"] = _problem(case, seed)
        s["engine"] = native.Engine(0, **_cfg(case))
        s["engine"].set_mesh(verts, tets)
    elif kind == "batch":
        probs = _instances(case, seed, case["instances"])
        s["sites"] = np.concatenate([p[2] for p in probs])
        s["engine"] = native.Engine(0, **_cfg(case))
        s["engine"].set_batch(probs)
    elif kind == "serve":
        u = meshgen.uniform24(21, case["jobs"])
        span = case["iters_hi"] - case["iters_lo"] + 1
        s["jobs"] = [(p, case["iters_lo"] + int(u[i] * span))
                     for i, p in enumerate(_instances(case, seed, case["jobs"]))]
        s["server"] = native.Server(0, budget_bytes=64 << 30, **_cfg(case))
    elif kind == "program":
        s["problem"] = _problem(case, seed)
        s["dir"] = tempfile.TemporaryDirectory()
    elif kind == "knn_dev":
        s["ref"] = torch.from_numpy(np.ascontiguousarray(_uniform(2 * seed, case["n_ref"]).T)).cuda()
        s["query"] = torch.from_numpy(np.ascontiguousarray(_uniform(2 * seed + 1, case["n_query"]).T)).cuda()
        s["index"] = torch.empty((case["k"], case["n_query"]), dtype=torch.int32, device="cuda")
    else:
        s["points"] = _uniform(2 * seed, case["n_ref"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "lloyd":
        e = s["engine"]
        e.set_sites(s["sites"])
        e.lloyd(case["iters"])
        return e.sites()
    if kind == "step":
        e = s["engine"]
        e.set_sites(s["sites"])
        e.knn_step()
        e.clip_step()
        moments = e.moments()
        e.update_step()
        return {"moments": moments, "sites": e.sites()}
    if kind == "batch":
        e = s["engine"]
        e.set_sites(s["sites"])
        e.lloyd_graph(case["iters"])
        return e.sites()
    if kind == "serve":
        srv = s["server"]
        ids = [srv.submit(*p, it) for p, it in s["jobs"]]
        while any(srv.step()):
            pass
        return [srv.result(j) for j in ids]
    if kind == "program":
        verts, tets, sites = s["problem"]
        return native.compute_clipped_voro_diagram(verts, tets, sites, nb_iter=case["iters"], tet_k=case["tk"],
                                                   out_dir=s["dir"].name, form=case["form"], accum=case["accum"],
                                                   moments=case["moments"], site_k=case["k"])
    if kind == "knn_dev":
        rc = native.lib().vd_knn_dev(s["ref"].data_ptr(), case["n_ref"], case["n_ref"], s["query"].data_ptr(),
                                     case["n_query"], case["n_query"], 3, case["k"], s["index"].data_ptr(),
                                     case["n_query"], None)
        if rc != native.VD_OK:
            raise RuntimeError("vd_knn_dev failed (%d)" % rc)
        return s["index"]
    kn = native.KnProblem(s["points"], case["k"])
    kn.solve()
    out = {"lists": kn.knearests(), "points": kn.points(), "permutation": kn.permutation()}
    kn.close()
    return out


# Arithmetic that an iteration cannot do without, per tet: distances to its
# candidates (8 operations each), and about 6 pieces (sites are about a tenth
# of the tets; denser sites make more), each some 10 determinants of 45
# operations for its cuts and 10 vertices of 545 for its volume and moments.
_PIECE = 10 * 45 + 10 * 545


def _iteration(n_verts, n_tets, n_sites, tk, k):
    tk = tk or max(20, 10 * math.ceil(8 * math.log10(7.0 * n_sites / max(n_tets, 1) + 1)))
    pieces = 6.0 * n_tets * max(1.0, 10.0 * n_sites / n_tets) ** (2.0 / 3.0)
    flops = 8.0 * (n_tets * tk + n_sites * k) + pieces * _PIECE
    return 12.0 * n_verts + 16.0 * n_tets + 24.0 * n_sites, flops


def work(case):
    kind = case["kind"]
    if kind in ("knn_dev", "kn"):
        out = 4 * case["n_query"] * case["k"]
        return {"bytes": 12 * case["n_ref"] + (12 * case["n_query"] if kind == "knn_dev" else 16 * case["n_ref"]) + out,
                "flops": 8 * case["n_query"] * case["k"]}
    if kind in ("batch", "serve"):
        n = case["instances"] if kind == "batch" else case["jobs"]
        iters = case["iters"] if kind == "batch" else 0.5 * (case["iters_lo"] + case["iters_hi"])
        parts = [((m + 1) ** 3, 6 * m ** 3, 6 * m ** 3 // 10, iters) for m in _sizes(case, n)]
    elif case["mesh"] == "torus":
        n_vox = 2 * math.pi ** 2 * 0.35 * 0.15 ** 2 * case["n"] ** 3
        parts = [(1.1 * n_vox, 6 * n_vox, case["n_sites"], case["iters"])]
    else:
        parts = [((case["n"] + 1) ** 3, 6 * case["n"] ** 3, case["n_sites"], case["iters"])]
    b = f = 0.0
    for nv, nt, ns, it in parts:
        pb, pf = _iteration(nv, nt, ns, case["tk"], case["k"])
        b, f = b + it * pb, f + it * pf
    if kind == "step":
        b += 32.0 * case["n_sites"]
    return {"bytes": b, "flops": f}


# ---- the same results in 64 bits, by cutting tets into tets ----------------

_EXACT_PAIRS = 7_000_000  # (tet, candidate) pairs over all iterations, at most


def _nearest(points, refs, k, skip_self):
    """k nearest refs of every point, nearest first (rows skip their own index when skip_self)."""
    rows = []
    step = max(1, 40_000_000 // max(1, refs.shape[0]))
    for a in range(0, points.shape[0], step):
        d = torch.cdist(points[a:a + step], refs, compute_mode="donot_use_mm_for_euclid_dist")
        if skip_self:
            i = torch.arange(d.shape[0])
            d[i, i + a] = math.inf
        rows.append(torch.topk(d, k, dim=1, largest=False, sorted=True).indices)
    return torch.cat(rows)


def _cut(p, f):
    """Pieces of the tets p (m,4,3) on the side f >= 0 of their planes (f: (m,4) values at
    the corners, with both signs in every row); returns the pieces and their source rows."""
    order = torch.argsort((f >= 0).to(torch.int8), dim=1, descending=True, stable=True)
    p = torch.gather(p, 1, order[:, :, None].expand(-1, -1, 3))
    f = torch.gather(f, 1, order)
    inside = (f >= 0).sum(1)
    out, src = [], []

    def mix(r, i, j):
        t = (f[r, i] / (f[r, i] - f[r, j]))[:, None]
        return p[r, i] + t * (p[r, j] - p[r, i])

    def put(r, *corners):
        out.append(torch.stack(corners, 1))
        src.append(r)

    r = torch.nonzero(inside == 1)[:, 0]
    put(r, p[r, 0], mix(r, 0, 1), mix(r, 0, 2), mix(r, 0, 3))
    for need, prism in ((2, lambda r: (p[r, 0], mix(r, 0, 2), mix(r, 0, 3), p[r, 1], mix(r, 1, 2), mix(r, 1, 3))),
                        (3, lambda r: (p[r, 0], p[r, 1], p[r, 2], mix(r, 0, 3), mix(r, 1, 3), mix(r, 2, 3)))):
        r = torch.nonzero(inside == need)[:, 0]
        a, b, c, d, e, g = prism(r)
        put(r, a, b, c, d)
        put(r, b, c, d, e)
        put(r, c, d, e, g)
    return torch.cat(out), torch.cat(src)


def _site_moments(verts, tets, sites, tk, k):
    """Per site (volume, first moments) of the tets' pieces in its cell, in 64 bits."""
    n_sites, k, tk = sites.shape[0], min(k, sites.shape[0] - 1), min(tk, sites.shape[0])
    corners = verts[tets]
    cand = _nearest(corners.mean(1), sites, tk, False)
    nbr = _nearest(sites, sites, k, True)
    total = torch.zeros((n_sites, 4), dtype=torch.float64)
    step = max(1, 1_000_000 // tk)
    for a in range(0, corners.shape[0], step):
        c = cand[a:a + step].reshape(-1)
        sums = torch.zeros((c.shape[0], 4), dtype=torch.float64)
        p = corners[a:a + step].repeat_interleave(tk, 0)
        pair = torch.arange(c.shape[0])

        def keep(p, pair):
            e = p[:, 1:] - p[:, :1]
            v = (e[:, 0] * torch.linalg.cross(e[:, 1], e[:, 2])).sum(1).abs() / 6.0
            sums.index_add_(0, pair, torch.cat([v[:, None], v[:, None] * p.mean(1)], 1))

        for j in range(k):
            if p.shape[0] == 0:
                break
            s = sites[c[pair]]
            z = sites[nbr[c[pair], j]]
            d = z - s
            r = p - s[:, None]
            f = 0.5 * (d * d).sum(1)[:, None] - (r * d[:, None]).sum(2)
            done = 4.0 * (r * r).sum(2).amax(1) < (d * d).sum(1)
            whole = (f >= 0).all(1)
            none = (f < 0).all(1)
            if bool(done.any()):
                keep(p[done], pair[done])
            part = ~done & ~whole & ~none
            stay = ~done & whole
            q, src = _cut(p[part], f[part])
            p, pair = torch.cat([p[stay], q]), torch.cat([pair[stay], pair[part][src]])
        keep(p, pair)
        sums[sums[:, 0] < 0.1] = 0.0  # pieces below 0.1 cubic units are not accumulated
        total.index_add_(0, c, sums)
    return total


def _exact_chain(verts, tets, sites, iters, tk, k):
    v = torch.from_numpy(verts).double()
    t = torch.from_numpy(tets).long()
    s = torch.from_numpy(sites).double()
    m = None
    for _ in range(iters):
        m = _site_moments(v, t, s, tk, k)
        some = m[:, 0] != 0
        s = torch.where(some[:, None], m[:, 1:] / torch.where(some, m[:, 0], torch.ones_like(m[:, 0]))[:, None], s)
    return m.numpy(), s.numpy()


def exact(case, seed):
    """Where the moments are the robust ones (the reference's decomposition is not the
    volume where a seed lies near a face plane) and the problem is small; else None."""
    if case["kind"] not in ("lloyd", "step") or case["moments"] != "robust" or not case["tk"] or case["mesh"] != "cube":
        return None
    if 6 * case["n"] ** 3 * case["tk"] * case["iters"] > _EXACT_PAIRS:
        return None
    verts, tets, sites = _problem(case, seed)
    m, s = _exact_chain(verts, tets, sites, case["iters"], case["tk"], case["k"])
    return {"moments": m, "sites": s} if case["kind"] == "step" else s
