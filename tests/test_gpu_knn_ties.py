"""The nearest-neighbour search where more points lie at the k-th distance than
its candidate list holds (20): places shared by thousands of points, as scans
have them that store each invalid sample as one repeated point, alone, with
nearer points beside them, and with points whose coordinates are NaN.

Coordinates are small integers, so float32 squared distances are exact and the
expected neighbours, ties to the lower index, are those of a brute-force search
in whole numbers: compared for equality.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cloud(kind, n, seed):
    r = np.random.RandomState(seed)
    p = r.randint(0, 64, (n, 3))
    p[:, 2] //= 16
    if kind == "one":  # two thirds of the points at one place, at indices spread over the cloud
        p[r.rand(n) < 2 / 3] = (31, 7, 1)
    elif kind == "all":
        p[:] = (3, 4, 5)
    elif kind == "ring":  # a few points in the middle of thousands at four places at one distance
        at = np.array([(20, 30, 2), (40, 30, 2), (30, 20, 2), (30, 40, 2)])
        p = at[r.randint(0, 4, n)]
        p[r.permutation(n)[:7]] = [(30, 30, 2)] * 4 + [(30, 31, 2), (31, 30, 2), (29, 29, 2)]
    return p


def _nearest(query, points, k, valid):
    out = np.empty((len(query), k), np.int64)
    at = np.nonzero(valid)[0]
    for b in range(0, len(query), 256):
        d = ((query[b:b + 256, None] - points[None, at]) ** 2).sum(-1)
        out[b:b + 256] = at[np.argsort(d * len(points) + at, axis=1)[:, :k]]
    return out


@pytest.mark.parametrize("kind,n,k,nan", [("one", 3000, 10, 0), ("one", 6001, 16, 0), ("one", 2500, 1, 0), ("all", 21, 16, 0),
                                          ("all", 1999, 10, 0), ("ring", 3000, 10, 0), ("ring", 2999, 6, 0), ("ring", 4000, 16, 5),
                                          ("one", 3000, 8, 40)])
def test_neighbours(pkg, kind, n, k, nan):
    import torch
    print("case", kind, n, k, nan, flush=True)
    p = _cloud(kind, n, n + k)
    rec = p.astype(np.float32)
    bad = np.random.RandomState(k).permutation(n)[:nan]
    rec[bad, 1] = np.nan
    valid = np.ones(n, bool)
    valid[bad] = False
    t = torch.from_numpy(rec).cuda()
    nrm, cur = torch.empty((n, 3), device="cuda"), torch.empty((n,), device="cuda")
    knn = torch.full((n, k), -1, dtype=torch.int32, device="cuda")
    ctx = pkg.PoissonReconstruction(depth=5)
    torch.cuda.synchronize()
    rc = pkg.binding.lib().psr_estimate_normals(ctx._ctx, t.data_ptr(), n, 12, k, (ctypes.c_float * 3)(0, 0, 0),
                                                nrm.data_ptr(), cur.data_ptr(), knn.data_ptr())
    assert rc == 0
    got = knn.cpu().numpy()
    ctx.close()
    assert np.array_equal(got[valid], _nearest(p[valid], p, k, valid))
    assert np.all(got[~valid] == 0x7fffffff)  # a point without a place has no nearest


@pytest.mark.parametrize("kind,n,nv", [("one", 3000, 300), ("ring", 2500, 77), ("all", 4000, 33)])
def test_colours(pkg, kind, n, nv):
    """Within 8 float32 roundings of a value below 1, as the four points and their exact squared distances give it."""
    import torch
    print("case", kind, n, nv, flush=True)
    r = np.random.RandomState(n)
    p = _cloud(kind, n, n)
    v = p[r.randint(0, n, nv)] + r.randint(-1, 2, (nv, 3))
    col = r.rand(n, 3).astype(np.float32)
    ctx = pkg.PoissonReconstruction(depth=5)
    got = ctx.VertexColors(torch.from_numpy(v.astype(np.float32)).cuda(), torch.from_numpy(p.astype(np.float32)).cuda(),
                           torch.from_numpy(col).cuda())
    ctx.close()
    near = _nearest(v, p, 4, np.ones(n, bool))
    d = ((v[:, None] - p[near]) ** 2).sum(-1).astype(np.float64)
    s = d.sum(1, keepdims=True)
    w = np.where(s > 0, d / np.where(s > 0, s, 1), 0.25)
    want = (w[..., None] * col[near].astype(np.float64)).sum(1)
    assert np.all(np.abs(got - want) <= 8 * 2.0 ** -24)
