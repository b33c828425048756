"""The workloads that the framework's speed is measured on.

Each case is one call of a public entry point as a user's program makes it:
a graph build (resident, allocation-free, or on host buffers), a label-filtered
or stitched build, or a batch of queries against a built graph. The vectors
are made on the GPU from the seed: Gaussian-mixture rows (L2-normalised for
float types, clip(round(64 + 24 z)) for uint8), or isotropic rows where
"centers" is 0.

Every output is a whole number (neighbour ids, degrees, entry points) or a
distance in the framework's canonical arithmetic, which fixes the order of
every sum, so a correct implementation gives the same bits: all tolerances are
exact.
"""
import heapq

import numpy as np
import torch

import dance_amd as D
from dance_amd import filtered as F

_DT = {"f32": D.DTYPE_F32, "u8": D.DTYPE_U8, "f16": D.DTYPE_F16}
_BYTES = {"f32": 4, "u8": 1, "f16": 2}


def listed():
    return [
        # The smallest call: one small segment indexed inside a serving loop,
        # through the entry that may not allocate. Latency and launches count.
        dict(name="build_small", op="build", entry="noalloc", kind="f32", n=2_000, dim=96, centers=0, R=32, L=64,
             C=48, STEPS=32),
        # 100k isotropic rows (no clusters: the hardest data for the search).
        dict(name="build_100k", op="build", entry="resident", kind="f32", n=100_000, dim=96, centers=0, R=64, L=100,
             C=80, STEPS=64),
        # One shard of the sharded pipeline: the v8 builder on host buffers,
        # upload and download included, with the pipeline's own degrees.
        dict(name="build_shard_host", op="build", entry="host_v8", kind="f32", n=250_000, dim=128, centers=256, R=42,
             L=100, C=84, STEPS=20),
        # The ordinary build: 1M clustered fp32 rows in HBM.
        dict(name="build_1m", op="build", entry="resident", kind="f32", n=1_000_000, dim=96, centers=256, R=64,
             L=100, C=80, STEPS=64),
        # The largest: the data no longer fits the Infinity Cache.
        dict(name="build_4m", op="build", entry="resident", kind="f32", n=4_000_000, dim=96, centers=256, R=64,
             L=100, C=80, STEPS=64),
        # uint8 rows (integer distances, many ties).
        dict(name="build_u8_2m", op="build", entry="resident", kind="u8", n=2_000_000, dim=128, centers=1024, R=64,
             L=100, C=80, STEPS=64),
        # fp16 rows at a ragged size and width, with a longer list than the
        # default (a quality setting).
        dict(name="build_f16_l150", op="build", entry="resident", kind="f16", n=300_007, dim=100, centers=256, R=64,
             L=150, C=96, STEPS=64),
        # The label-filtered build: 1-8 Zipf labels per row.
        dict(name="filtered_u8", op="filtered", kind="u8", n=250_000, dim=192, centers=1024, R=64, L=100, vocab=5_000,
             labels=8),
        # The stitched build: one label per row, per-label graphs.
        dict(name="stitched_u8", op="stitched", kind="u8", n=500_000, dim=192, centers=1024, R=32, L=100, C=96,
             STEPS=64, nlabels=50),
        # A large batch of queries (offline scoring, recall measurement).
        dict(name="search_10k", op="search", kind="f32", n=1_000_000, dim=96, centers=256, R=64, L=100, C=80,
             STEPS=64, nq=10_000, k=10, SL=100, vocab=0, labels=0),
        # A handful of queries: what one serving request brings.
        dict(name="search_16", op="search", kind="f32", n=200_000, dim=96, centers=256, R=64, L=100, C=80, STEPS=64,
             nq=16, k=10, SL=50, vocab=0, labels=0),
        # Label-filtered queries over a filtered graph.
        dict(name="search_filtered_1k", op="search", kind="u8", n=100_000, dim=192, centers=1024, R=64, L=100, C=0,
             STEPS=64, nq=1_000, k=10, SL=100, vocab=2_000, labels=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["build", "build", "build", "build", "filtered", "stitched", "search", "search"])
    kind = rng.choice(["f32", "f32", "u8", "f16"])
    dim = {"f32": rng.randint(24, 200), "f16": rng.randint(24, 256), "u8": rng.randint(32, 256)}[kind]
    centers = rng.choice([0, 64, 256, 1024])
    if op == "build":
        entry = rng.choice(["resident", "resident", "host", "host_v8", "noalloc"])
        R = rng.choice([32, 42, 48, 64])
        L = rng.randint(max(50, R), 200)
        n = _log_int(rng, 1_000, 60_000 if entry == "noalloc" else 600_000 if centers == 0 else 1_200_000)
        if entry != "resident" and kind == "f16":
            kind = "f32"  # the host entries take fp32 and uint8 rows
        if entry == "noalloc":
            n = min(n, 50_000)  # the library's scratch array bounds it
        return dict(op=op, entry=entry, kind=kind, n=n, dim=dim, centers=centers, R=R, L=L,
                    C=rng.randint(R, 2 * R) if R < 64 else rng.randint(64, 128), STEPS=rng.randint(16, 64))
    if op == "filtered":
        if kind == "f32":
            kind = "u8"
        return dict(op=op, kind=kind, n=_log_int(rng, 3_000, 250_000), dim=dim, centers=centers,
                    R=rng.choice([32, 48, 64]), L=rng.randint(64, 120), vocab=_log_int(rng, 50, 5_000),
                    labels=rng.randint(1, 8))
    if op == "stitched":
        R = rng.choice([24, 32, 48])
        return dict(op=op, kind=kind, n=_log_int(rng, 10_000, 500_000), dim=dim, centers=centers, R=R,
                    L=rng.randint(64, 128), C=rng.randint(2 * R, 3 * R), STEPS=rng.randint(24, 64),
                    nlabels=_log_int(rng, 4, 60))
    filt = rng.random() < 0.3
    if filt and kind == "f32":
        kind = "u8"
    k = rng.choice([1, 10, 10, 50])
    return dict(op=op, kind=kind, n=_log_int(rng, 5_000, 100_000 if filt else 500_000), dim=dim, centers=centers,
                R=64, L=100, C=0 if filt else 80, STEPS=64, nq=_log_int(rng, 1, 10_000), k=k,
                SL=_log_int(rng, max(k, 10), 400), vocab=_log_int(rng, 20, 2_000) if filt else 0,
                labels=rng.randint(1, 8) if filt else 0)


def _rows(kind, n, dim, centers, gen, cent=None):
    """n rows on the GPU and the centers they are drawn around."""
    if centers and cent is None:
        cent = torch.randn(centers, dim, device="cuda", generator=gen)
    x = torch.randn(n, dim, device="cuda", generator=gen)
    if centers:
        x = cent[torch.randint(0, centers, (n,), device="cuda", generator=gen)] + 0.3 * x
    if kind == "u8":
        return torch.clamp(torch.round(64 + 24 * x), 0, 255).to(torch.uint8), cent
    x = x / x.norm(dim=1, keepdim=True)
    return (x.half() if kind == "f16" else x).contiguous(), cent


def _global_start(x):
    """The row nearest to the centroid."""
    m = x.float().mean(dim=0)
    best, at = None, 0
    for b in range(0, x.shape[0], 1 << 18):
        d = ((x[b:b + (1 << 18)].float() - m) ** 2).sum(1)
        v, i = d.min(0)
        if best is None or v.item() < best:
            best, at = v.item(), b + int(i)
    return at


def _out(n, width):
    return (torch.empty(n, width, dtype=torch.int32, device="cuda"), torch.empty(n, dtype=torch.int32, device="cuda"))


def _label_state(case, seed):
    ls = F.synth_labels(case["n"], case["vocab"], 1, min(case["labels"], case["vocab"]), 1.0, seed=seed)
    return ls, F.balanced_label_starts(ls)


def _filtered_build(st, case):
    F.filtered_build_resident(st["x"].data_ptr(), _DT[case["kind"]], case["n"], case["dim"], st["ls"], st["starts"],
                              case["R"], case["L"], case["L"], F.DISKANN_MAXC, 64, 1.2, D.INVALID, st["gstart"],
                              st["graph"].data_ptr(), st["degree"].data_ptr())


def _resident_build(st, case):
    D.vamana_build_resident(st["x"].data_ptr(), _DT[case["kind"]], case["n"], case["dim"], case["R"], case["L"],
                            case["C"], case["STEPS"], st["graph"].data_ptr(), st["degree"].data_ptr())


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n, dim = case["n"], case["dim"]
    x, cent = _rows(case["kind"], n, dim, case["centers"], gen)
    st = {"case": case, "x": x}
    op = case["op"]
    if op == "build":
        if case["entry"].startswith("host"):
            st["x"] = x.cpu().numpy()
        else:
            st["graph"], st["degree"] = _out(n, case["R"])
    elif op == "filtered":
        st["ls"], st["starts"] = _label_state(case, seed)
        st["gstart"] = _global_start(x)
        st["graph"], st["degree"] = _out(n, case["R"])
    elif op == "stitched":
        lab = torch.randint(0, case["nlabels"], (n,), device="cuda", generator=gen)
        st["points"] = torch.argsort(lab, stable=True).cpu().numpy().astype(np.uint32)
        off = np.zeros(case["nlabels"] + 1, np.uint32)
        off[1:] = np.cumsum(torch.bincount(lab, minlength=case["nlabels"]).cpu().numpy())
        st["offsets"] = off
        st["graph"], st["degree"] = _out(n, case["R"])
    else:
        q, _ = _rows(case["kind"], case["nq"], dim, case["centers"], gen, cent)
        st["q"] = q.cpu().numpy()
        st["graph"], st["degree"] = _out(n, case["R"])
        st["label_args"] = (None, None, None)
        if case["vocab"]:
            st["ls"], st["starts"] = _label_state(case, seed)
            st["gstart"] = _global_start(x)
            _filtered_build(st, case)
            # each query asks for the label of some row, so frequent labels are asked for more often
            pick = np.random.default_rng(seed + 1).integers(0, st["ls"].labels.shape[0], case["nq"])
            ql = st["ls"].labels[pick]
            st["label_args"] = (st["ls"].offsets, st["ls"].labels, ql)
            st["start"] = st["starts"][ql]
        else:
            _resident_build(st, case)
            st["start"] = D.last_medoid()
    return st


def run(st):
    case = st["case"]
    op, n, dim = case["op"], case["n"], case["dim"]
    if op == "build":
        if case["entry"].startswith("host"):
            r = D.vamana_build(st["x"], case["R"], case["L"], case["C"], case["STEPS"],
                               entry="v8" if case["entry"] == "host_v8" else "vnew2")
            return {"graph": r.graph, "degree": r.degree, "medoid": r.medoid}
        if case["entry"] == "noalloc":
            D.vamana_build_resident_noalloc(st["x"].data_ptr(), _DT[case["kind"]], n, dim, case["R"], case["L"],
                                            case["C"], case["STEPS"], st["graph"].data_ptr(),
                                            st["degree"].data_ptr())
        else:
            _resident_build(st, case)
        return {"graph": st["graph"], "degree": st["degree"], "medoid": D.last_medoid()}
    if op == "filtered":
        _filtered_build(st, case)
        return {"graph": st["graph"], "degree": st["degree"]}
    if op == "stitched":
        med = D.stitched_build_resident(st["x"].data_ptr(), _DT[case["kind"]], n, dim, st["offsets"], st["points"],
                                        case["R"], case["L"], case["C"], case["STEPS"], 64, case["R"],
                                        st["graph"].data_ptr(), st["degree"].data_ptr())
        return {"graph": st["graph"], "degree": st["degree"], "medoids": med}
    ids, dists = D.search_resident(st["x"].data_ptr(), _DT[case["kind"]], n, dim, st["graph"].data_ptr(),
                                   st["degree"].data_ptr(), case["R"], st["start"], st["q"], case["k"], case["SL"],
                                   *st["label_args"])
    return {"ids": ids, "dists": dists}


def work(case):
    """Each row read and each output written once; three operations per
    dimension (difference, multiply-add) of each distance that the algorithm
    asks for. About 20 of an expansion's neighbours are new on clustered
    rows; a build searches every row in four iterations (a label-filtered one
    in three rounds, over the rows of its labels), a query expands about L
    entries."""
    row, n = case["dim"] * _BYTES[case["kind"]], case["n"]
    per = 3 * case["dim"]
    if case["op"] == "search":
        dist = case["nq"] * case["SL"] * 20
        return {"bytes": case["nq"] * (row + 8 * case["k"]) + dist * row, "flops": dist * per}
    if case["op"] == "filtered":
        dist = n * 3 * 64 * 20
    else:
        dist = n * 4 * min(case["STEPS"], case["L"]) * 20
    return {"bytes": n * (row + 4 * case["R"] + 4), "flops": dist * per}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The queries' distances in 64 bits: a best-first search with a list of
    SL entries over the same graph. Graphs are ids and have no such value."""
    if case["op"] != "search" or case["nq"] > 1_000:
        return None
    st = prepare(case, seed)
    x, q = st["x"].cpu().numpy().astype(np.float64), st["q"].astype(np.float64)
    graph, degree = st["graph"].cpu().numpy(), st["degree"].cpu().numpy()
    off, lab, ql = st["label_args"]
    start = np.broadcast_to(np.asarray(st["start"], np.int64), (case["nq"],))
    out = np.full((case["nq"], case["k"]), float(np.finfo(np.float32).max))

    def dist(i, ids):
        t = x[ids] - q[i]
        return (t * t).sum(1)

    for i in range(case["nq"]):
        s = int(start[i])
        seen = {s}
        best = [(float(dist(i, [s])[0]), s)]  # the list, nearest first
        todo = list(best)
        while todo:
            d, u = heapq.heappop(todo)
            if len(best) >= case["SL"] and (d, u) > best[-1]:
                break
            new = [v for v in graph[u, :degree[u]].tolist() if v not in seen
                   and (ql is None or ql[i] in lab[off[v]:off[v + 1]])]
            seen.update(new)
            if not new:
                continue
            found = list(zip(dist(i, new).tolist(), new))
            if len(best) >= case["SL"]:
                found = [f for f in found if f < best[-1]]
            for f in found:
                heapq.heappush(todo, f)
            best = sorted(best + found)[:case["SL"]]
        for j, (d, _) in enumerate(best[:case["k"]]):
            out[i, j] = d
    return {"ids": None, "dists": out}
