"""Edges of the kernels' tiles and dispatch rules, against the CPU oracle bit
for bit (gfx950 only): sizes around a workgroup's share, widths of every
compiled row group, and both sides of each rule that picks a kernel."""
import numpy as np
import pytest

import dance_amd as D
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rows(kind, n, dim, seed=3, centers=0):
    rng = np.random.default_rng(seed)
    if kind == "u8":
        return rng.integers(0, 256, (n, dim), dtype=np.uint8)
    x = rng.standard_normal((n, dim))
    if centers:
        x = 0.3 * x + rng.standard_normal((centers, dim))[rng.integers(0, centers, n)]
    x /= np.linalg.norm(x, axis=1, keepdims=True)
    return x.astype(np.float16 if kind == "f16" else np.float32)


# candidates per workgroup 4 / 2 / 1 by row width; samples in strides of 64
@pytest.mark.parametrize("kind,dim", [("f32", 20), ("f32", 128), ("f32", 200), ("f32", 500), ("u8", 130), ("f16", 77),
                                      ("f16", 801)])
@pytest.mark.parametrize("n", [2, 5, 65, 1023, 4097])
def test_medoid_group_edges(kind, dim, n):
    x = rows(kind, n, dim)
    if kind == "f32" and n > 5:
        x[n // 2] = np.inf  # scores that are NaN or inf
        x[n // 3, 1] = np.nan
    gm, gs, gc = D.stage_medoid(x)
    om, os_, oc = O.medoid(x)
    assert np.array_equal(gc, oc)
    same = gs.view(np.uint32) == os_.view(np.uint32)
    assert np.all(same | (np.isnan(gs) & np.isnan(os_)))
    assert gm == om


# u8 rows of 1, 2, 4 and 8 chunks per lane take the schedule's MFMA cells; 4095
# and 4096 rows are the two sides of the rule that needs 16 cells of 256 rows
@pytest.mark.parametrize("n,dim", [(4095, 40), (4096, 40), (4097, 129), (5000, 300), (4500, 600)])
def test_u8_schedule_widths(n, dim):
    x = rows("u8", n, dim)
    og, od, om = O.vnew2_build(x, 24, 48, 32, 24)
    r = D.vamana_build(x, 24, 48, 32, 24)
    assert r.medoid == om
    assert np.array_equal(r.degree, od) and np.array_equal(r.graph, og)


# rows without clusters: from 4 MiB of (padded) rows on every iteration takes the
# code-row bound; the same rows below it, and clustered rows, keep 1 and 2 exact
@pytest.mark.parametrize("n,centers,middle", [(11_000, 0, True), (10_900, 0, False), (11_000, 40, False)])
def test_bound_in_every_iteration_of_dense_data(n, centers, middle):
    x = rows("f32", n, 96, centers=centers)
    assert (n * 384 > 4 << 20) == (n == 11_000)
    og, od, om = O.vnew2_build(x, 48, 64, 64, 32)
    r = D.vamana_build(x, 48, 64, 64, 32)
    assert r.medoid == om
    assert np.array_equal(r.degree, od) and np.array_equal(r.graph, og)
    checks = r.kernel_profile["bound_checks_iter"]
    assert checks[0] > 0
    assert [c > 0 for c in checks[1:3]] == [middle, middle]


# code rows of two chunk groups: widths on both sides of 112, 128 and 240
# dimensions and of each compiled row group, pools of 2 and 4 slots per lane
@pytest.mark.parametrize("kind,dim,L", [("f32", 113, 64), ("f32", 128, 140), ("f32", 129, 64), ("f32", 240, 64),
                                        ("f32", 241, 64), ("f16", 113, 64), ("f16", 128, 64), ("f16", 191, 140),
                                        ("f16", 192, 64), ("f16", 240, 64), ("f16", 241, 64)])
@pytest.mark.parametrize("centers", [0, 20])
def test_wide_code_rows(kind, dim, L, centers):
    import torch
    n, R, C, steps = 4000, 32, 48, 32
    x = rows(kind, n, dim, centers=centers)
    x[5:9] = x[4]  # equal rows
    x[30] *= 100 if kind == "f32" else 4
    if centers == 0:
        x[11] = np.inf
        x[12, 3] = np.nan
    og, od, om = O.vnew2_build(x, R, L, C, steps)
    xt = torch.from_numpy(x).cuda()
    g = torch.empty((n, R), dtype=torch.int32, device="cuda")
    d = torch.empty((n,), dtype=torch.int32, device="cuda")
    D.vamana_build_resident(xt.data_ptr(), D.dtype_code(x), n, dim, R, L, C, steps, g.data_ptr(), d.data_ptr())
    assert D.last_medoid() == om
    assert np.array_equal(d.cpu().numpy().view(np.uint32), od)
    assert np.array_equal(g.cpu().numpy().view(np.uint32), og)
    assert (D.last_kernel_profile()["bound_checks"] > 0) == (dim <= 240)


# base rows read packed: row lengths that leave a last chunk of 1 to 15 bytes,
# rows that start at any byte, both sides of the rule (one query and many),
# pools of 1 and 2 slots per lane and beyond, and rows too wide for it
@pytest.mark.parametrize("kind,dim", [("u8", 1), ("u8", 15), ("u8", 17), ("u8", 99), ("u8", 131), ("u8", 509), ("u8", 513),
                                      ("f16", 7), ("f16", 101), ("f16", 130), ("f32", 3), ("f32", 33), ("f32", 97),
                                      ("f32", 127), ("f32", 130)])
@pytest.mark.parametrize("shift,nq,L", [(0, 1, 10), (1, 2, 65), (5, 1, 129), (0, 200, 20)])
def test_packed_base_rows(kind, dim, shift, nq, L):
    import torch
    n, R, k = 5000, 16, 10
    x = rows(kind, n, dim, seed=dim)
    qs = rows(kind, nq, dim, seed=dim + 1)
    if kind != "u8":
        x[17] = np.inf
    rng = np.random.default_rng(dim)
    graph = rng.integers(0, n, (n, R), dtype=np.uint32)
    degree = rng.integers(0, R + 1, n).astype(np.uint32)
    starts = np.array([7], np.uint32)
    want = O.query_search(x, graph, degree, starts, qs, k, L)
    shift -= shift % x.itemsize if kind != "u8" else 0  # elements stay aligned
    flat = torch.zeros(x.nbytes + 64, dtype=torch.uint8, device="cuda")
    flat[shift:shift + x.nbytes] = torch.from_numpy(x.reshape(-1).view(np.uint8)).cuda()
    g, d = torch.from_numpy(graph.view(np.int32)).cuda(), torch.from_numpy(degree.view(np.int32)).cuda()
    got = D.search_resident(flat.data_ptr() + shift, D.dtype_code(x), n, dim, g.data_ptr(), d.data_ptr(), R, starts, qs,
                            k, L)
    for a in (got, D.search(x, graph, degree, starts, qs, k, L)):
        assert np.array_equal(a[0], want[0])
        assert np.array_equal(a[1].view(np.uint32), want[1].view(np.uint32))


# calls of different sizes share leased memory, also from several threads at a
# time and after a call that fails with its lease open
def test_leased_memory_reuse():
    import threading
    import torch
    dims, R, k = (33, 96, 200, 17), 16, 10
    cases = []
    for i, dim in enumerate(dims):
        n = 1500 + 700 * i
        x, qs = rows("f32", n, dim, seed=i), rows("f32", 5 + 60 * i, dim, seed=i + 9)
        og, od, om = O.vnew2_build(x, R, 32, 24, 16)
        cases.append((x, qs, og, od, O.query_search(x, og, od, om, qs, k, 40), om))
    errors = []

    def work(t):
        try:
            for r in range(6):
                x, qs, og, od, want, om = cases[(r + t) % len(cases)]
                n, dim = x.shape
                ids, dd = D.search(x, og, od, om, qs, k, 40)
                assert np.array_equal(ids, want[0]) and np.array_equal(dd, want[1])
                if r % 2 == t % 2:
                    xt = torch.from_numpy(x).cuda()
                    g = torch.empty((n, R), dtype=torch.int32, device="cuda")
                    d = torch.empty((n,), dtype=torch.int32, device="cuda")
                    torch.cuda.synchronize()
                    D.vamana_build_resident(xt.data_ptr(), D.dtype_code(x), n, dim, R, 32, 24, 16, g.data_ptr(),
                                            d.data_ptr())
                    assert np.array_equal(g.cpu().numpy().view(np.uint32), og)
                wide = np.zeros((4, 3000), np.float32)  # beyond the supported row width
                with pytest.raises(Exception):
                    D.search(wide, np.zeros((4, 2), np.uint32), np.ones(4, np.uint32), 0, wide[:1], 1, 4)
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


# small labels built together: empty labels, labels of one row and around a
# wave, a label too large for a group between them, pools on both sides of 128
@pytest.mark.parametrize("kind,dim,L", [("u8", 192, 64), ("f32", 96, 64), ("f32", 130, 140), ("f16", 77, 64)])
def test_stitched_label_groups(kind, dim, L):
    big = (4 << 20) // {"u8": 256, "f32": 384 if dim == 96 else 1024, "f16": 256}[kind] + 1  # its rows exceed 4 MiB
    sizes = [0, 1, 2, 63, 64, 65, 1500, 0, big, 300, 3, 1, 0]
    R, C, steps = 16, 24, 16
    n = sum(sizes)
    x = rows(kind, n, dim, centers=30)
    x[70:74] = x[69]
    rng = np.random.default_rng(dim)
    pts = rng.permutation(n).astype(np.uint32)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    for a, b in zip(off[:-1], off[1:]):
        pts[a:b] = np.sort(pts[a:b])
    g, d, med, st = D.stitched_build(x, off, pts, R, L, C, steps, R)
    for a, b, m in zip(off[:-1], off[1:], med):
        ids = pts[a:b]
        if a == b:
            assert m == D.INVALID
            continue
        og, od, om = O.vnew2_build(np.ascontiguousarray(x[ids]), R, L, C, steps)
        assert m == ids[om]
        for i in range(b - a):
            want = [ids[v] for v in og[i, :od[i]] if v < b - a and v != i]
            want = list(dict.fromkeys(want))
            assert d[ids[i]] == len(want) and g[ids[i], :len(want)].tolist() == want


# uint8 prunes from Gram tiles: rows of 1 to 16 chunks per lane, reverse lists on
# both sides of 128 entries, rows of more than 32 labels (no label masks), data
# full of equal rows and distances
@pytest.mark.parametrize("dim,R,C,labels,equal", [(7, 32, 64, 3, False), (130, 64, 750, 3, False),
                                                  (192, 64, 750, 40, False), (300, 32, 64, 3, True),
                                                  (513, 32, 64, 3, False), (1100, 16, 40, 3, True)])
def test_filtered_gram_prune(dim, R, C, labels, equal):
    from dance_amd import filtered as F
    n, vocab = 1200, 60 if labels > 32 else 6
    rng = np.random.default_rng(dim)
    x = rng.integers(0, 256, (n, dim), dtype=np.uint8)
    if equal:
        x = np.ascontiguousarray(x[rng.integers(0, 40, n)])
    ls = F.canonical_labels([rng.choice(vocab, labels, replace=False).tolist() for _ in range(n)], vocab)
    starts, gs = F.label_starts(x, ls), F.global_start(x)
    g, d = np.empty((n, R), np.uint32), np.empty(n, np.uint32)
    rc = F.build_rc(x, ls, starts, R, 48, 32, C, 24, 1.2, D.INVALID, gs, 2, graph=g, degree=d)
    orc, og, od, _ = O.filtered_build(x, ls.offsets, ls.labels, starts, ls.num_labels, R, 48, 32, C, 24, 1.2,
                                      D.INVALID, gs, 2, 0)
    assert rc == orc == 0
    assert np.array_equal(d, od) and np.array_equal(g, og)


# odd fp16 rows, whose last element is summed on its own: every row group, both
# sides of 240 dimensions, with the default degrees (batches of any size up to
# 64), pools of 2 and 4 slots per lane
@pytest.mark.parametrize("dim,L", [(63, 100), (127, 100), (129, 100), (129, 140), (191, 100), (193, 100), (239, 140),
                                   (241, 100), (255, 100), (301, 100), (513, 100)])
def test_odd_f16_builds(dim, L):
    import torch
    n, R, C, steps = 400, 64, 80, 24
    x = rows("f16", n, dim, seed=dim)
    og, od, om = O.vnew2_build(x, R, L, C, steps)
    xt = torch.from_numpy(x).cuda()
    g = torch.empty((n, R), dtype=torch.int32, device="cuda")
    d = torch.empty((n,), dtype=torch.int32, device="cuda")
    D.vamana_build_resident(xt.data_ptr(), D.dtype_code(x), n, dim, R, L, C, steps, g.data_ptr(), d.data_ptr())
    assert D.last_medoid() == om
    assert np.array_equal(d.cpu().numpy().view(np.uint32), od)
    assert np.array_equal(g.cpu().numpy().view(np.uint32), og)


# dense rows take the bound after the first iteration only where a row has more
# 128-byte lines than its code row: 64 fp16 dimensions have 1 and 1, 128 have 2 and
# 2, 80 have 2 and 1; the graphs are those of the exact searches
@pytest.mark.parametrize("dim,middle", [(64, False), (80, True), (128, False)])
def test_dense_rule_compares_lines(dim, middle, monkeypatch):
    import torch
    n, R = 34_000, 48
    x = torch.from_numpy(rows("f16", n, dim)).cuda()
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("DANCE_QBOUND", "0")
        g = torch.empty((n, R), dtype=torch.int32, device="cuda")
        d = torch.empty((n,), dtype=torch.int32, device="cuda")
        D.vamana_build_resident(x.data_ptr(), D.DTYPE_F16, n, dim, R, 64, 64, 40, g.data_ptr(), d.data_ptr())
        out.append((g, d))
        if not off:
            checks = D.last_kernel_profile()["bound_checks_iter"]
            assert checks[0] > 0
            assert [c > 0 for c in checks[1:3]] == [middle, middle]
            assert middle or checks[3] == 0
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


# the last iteration's bound on data without clusters whose long candidate rows
# keep the prune below a quarter of its pairs: most of a row's neighbours are new
@pytest.mark.parametrize("centers,last", [(0, True), (40, False)])
def test_last_iteration_bound_with_long_candidate_rows(centers, last, monkeypatch):
    import torch
    n, dim, R = 40_000, 96, 48
    x = torch.from_numpy(rows("f32", n, dim, centers=centers)).cuda()
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("DANCE_QBOUND", "0")
        g = torch.empty((n, R), dtype=torch.int32, device="cuda")
        d = torch.empty((n,), dtype=torch.int32, device="cuda")
        D.vamana_build_resident(x.data_ptr(), D.DTYPE_F32, n, dim, R, 100, 90, 40, g.data_ptr(), d.data_ptr())
        out.append((g, d))
        if not off:
            checks = D.last_kernel_profile()["bound_checks_iter"]
            assert [c > 0 for c in checks[:4]] == [True, False, False, last]
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


# later iterations take the bound only where a search meets enough candidates for its
# pool: few steps, short rows, a wide pool and small rows do without
@pytest.mark.parametrize("n,dim,R,L,C,steps,between,last", [
    (47_000, 79, 24, 162, 48, 33, False, False),
    (47_000, 79, 24, 84, 48, 33, True, False),
    (47_000, 96, 64, 162, 100, 20, False, False),
    (20_000, 96, 48, 100, 90, 40, False, False),
    (47_000, 79, 42, 84, 77, 33, False, True),
])
def test_later_bounds_need_candidates(n, dim, R, L, C, steps, between, last, monkeypatch):
    import torch
    x = torch.from_numpy(rows("f32", n, dim)).cuda()
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("DANCE_QBOUND", "0")
        g = torch.empty((n, R), dtype=torch.int32, device="cuda")
        d = torch.empty((n,), dtype=torch.int32, device="cuda")
        D.vamana_build_resident(x.data_ptr(), D.DTYPE_F32, n, dim, R, L, C, steps, g.data_ptr(), d.data_ptr())
        out.append((g, d))
        if not off:
            checks = D.last_kernel_profile()["bound_checks_iter"]
            assert [c > 0 for c in checks[:4]] == [True, between, between, last]
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


# what the calls keep is given back on request, and the next calls run
def test_release_memory():
    import torch
    n, dim, R = 100_000, 96, 16
    x = rows("f32", n, dim)
    rng = np.random.default_rng(0)
    graph, degree = rng.integers(0, n, (n, R), dtype=np.uint32), np.full(n, R, np.uint32)

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    D.release_memory()
    before = used()
    want = D.search(x, graph, degree, 0, x[:20], 10, 40)  # host rows: leases all of them
    assert used() - before > n * dim * 4
    D.release_memory()
    assert used() - before < 16 << 20
    got = D.search(x, graph, degree, 0, x[:20], 10, 40)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


# a search leases what it allocates: queries over large resident rows hold no copy
# of them, be they read as they are (96 dimensions) or packed (97)
@pytest.mark.parametrize("dim", [96, 97])
def test_small_search_leases_little(dim):
    import torch
    n, R = 200_000, 16
    x = torch.rand(n, dim, device="cuda")
    g = torch.randint(0, n, (n, R), dtype=torch.int32, device="cuda")
    d = torch.full((n,), R, dtype=torch.int32, device="cuda")
    q = np.ones((16, dim), np.float32)

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    D.release_memory()
    before = used()
    D.search_resident(x.data_ptr(), D.DTYPE_F32, n, dim, g.data_ptr(), d.data_ptr(), R, 0, q, 10, 50)
    assert used() - before < 16 << 20


# a call during a stream capture ends before it launches anything (it would wait
# for its stream, which a capture forbids), and the next call runs
CAPTURE = """
import ctypes
import numpy as np
import dance_amd as D
D.lib()
hip = ctypes.CDLL("libamdhip64.so")
n, dim, R = 2000, 96, 32
x = np.random.default_rng(0).standard_normal((n, dim)).astype(np.float32)
r = D.vamana_build(x, R, 64, 48, 32)
def build():
    return D.vamana_build(x, R, 64, 48, 32)
def search():
    return D.search(x, r.graph, r.degree, r.medoid, x[:4], 5, 20)[0]
want = search()
stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
for call in (build, search):
    assert hip.hipStreamBeginCapture(stream, 0) == 0  # global: no thread may wait
    try:
        call()
        refused = False
    except D.BuildError:
        refused = True
    hip.hipStreamEndCapture(stream, ctypes.byref(graph))
    hip.hipGetLastError()
    assert refused
assert np.array_equal(search(), want) and np.array_equal(build().graph, r.graph)
print("done")
"""


def test_calls_during_a_capture():
    import os
    import subprocess
    import sys
    r = subprocess.run([sys.executable, "-c", CAPTURE], cwd=os.path.dirname(os.path.dirname(D.__file__)), timeout=100,
                       capture_output=True, text=True)
    assert r.returncode == 0 and "done" in r.stdout, r.stderr[-2000:]
    assert r.stderr.count("cannot run during a stream capture") == 2, r.stderr[-2000:]


# uint8 prunes from Gram tiles at 8 and 16 chunks per lane, candidate rows of fewer
# and more than a wave
@pytest.mark.parametrize("dim", [600, 1100])
@pytest.mark.parametrize("R,C", [(16, 24), (24, 63), (48, 90)])
def test_wide_u8_prunes(dim, R, C):
    x = rows("u8", 700, dim)
    og, od, om = O.vnew2_build(x, R, 48, C, 24)
    r = D.vamana_build(x, R, 48, C, 24)
    assert r.medoid == om
    assert np.array_equal(r.degree, od) and np.array_equal(r.graph, og)
