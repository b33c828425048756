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
