"""The exact nearest-neighbour search behind the point normals and the vertex
colours, where its grid and lists can go wrong: few points, k at the ends of
each list length, points sharing a place (more ties at the k-th distance than
the candidate list holds), strided records, a cloud far from the origin.

Coordinates are small integers (times a power of two), so float32 squared
distances are exact and the expected neighbours, ties to the lower index, are
those of a brute-force search in whole numbers: compared for equality.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lattice(n, span, seed):
    """n points of an integer lattice, on a plane-like sheet: many equal distances and shared places."""
    r = np.random.RandomState(seed)
    p = r.randint(0, span, (n, 3))
    p[:, 2] = p[:, 2] * 3 // span
    return p


def _nearest(query, points, k):
    out = np.empty((len(query), k), np.int64)
    for b in range(0, len(query), 512):
        d = ((query[b:b + 512, None].astype(np.int64) - points[None].astype(np.int64)) ** 2).sum(-1)
        out[b:b + 512] = np.argsort(d * len(points) + np.arange(len(points)), axis=1)[:, :k]
    return out


@pytest.mark.parametrize("n,span,k,shift,stride", [
    (8, 4, 1, 0, 12), (5, 3, 16, 0, 12), (63, 8, 6, 0, 12), (64, 8, 8, 0, 20), (65, 2, 10, 0, 12),
    (1000, 40, 9, 0, 12), (1025, 5, 10, 512, 64), (3001, 100, 11, 0, 12), (5000, 60, 16, 256, 12), (4097, 3, 16, 0, 12)])
def test_neighbours_equal_brute_force(pkg, n, span, k, shift, stride):
    import torch
    print("case", n, span, k, shift, stride, flush=True)
    p = _lattice(n, span, n + k) + shift
    rec = np.zeros((n, stride // 4), np.float32)
    rec[:, :3] = p
    t = torch.from_numpy(rec).cuda()
    nrm, cur = torch.empty((n, 3), device="cuda"), torch.empty((n,), device="cuda")
    knn = torch.full((n, k), -1, dtype=torch.int32, device="cuda")
    ctx = pkg.PoissonReconstruction(depth=5)
    torch.cuda.synchronize()
    rc = pkg.binding.lib().psr_estimate_normals(ctx._ctx, t.data_ptr(), n, stride, k, (ctypes.c_float * 3)(0, 0, 0),
                                                nrm.data_ptr(), cur.data_ptr(), knn.data_ptr())
    assert rc == 0
    got = knn.cpu().numpy()
    ctx.close()
    kk = min(k, n)
    assert np.array_equal(got[:, :kk], _nearest(p, p, kk))
    assert np.all(got[:, kk:] == -1)


@pytest.mark.parametrize("n,nv,span", [(1, 3, 2), (3, 1, 4), (17, 100, 4), (2000, 999, 30), (3000, 65, 3)])
def test_colours_equal_brute_force(pkg, n, nv, span):
    """The weighted sum of the four expected neighbours' colours (weights from exact squared distances), within 8
    float32 roundings of a value below 1."""
    import torch
    print("case", n, nv, span, flush=True)
    r = np.random.RandomState(n)
    p, v = _lattice(n, span, n), r.randint(-2, span + 2, (nv, 3))
    col = r.rand(n, 3).astype(np.float32)
    ctx = pkg.PoissonReconstruction(depth=5)
    got = ctx.VertexColors(torch.from_numpy(v.astype(np.float32)).cuda(), torch.from_numpy(p.astype(np.float32)).cuda(),
                           torch.from_numpy(col).cuda())
    ctx.close()
    kk = min(4, n)
    near = _nearest(v, p, kk)
    d = ((v[:, None] - p[near]) ** 2).sum(-1).astype(np.float64)
    s = d.sum(1, keepdims=True)
    w = np.where(s > 0, d / np.where(s > 0, s, 1), 1.0 / kk)
    want = (w[..., None] * col[near].astype(np.float64)).sum(1)
    assert np.all(np.abs(got - want) <= 8 * 2.0 ** -24)


def test_non_finite_bounds_are_refused(pkg):
    import torch
    ctx = pkg.PoissonReconstruction(depth=5)
    xyz = torch.rand((1000, 3)).cuda()
    xyz[77, 1] = float("inf")
    with pytest.raises(pkg.binding.PsrError):
        ctx.EstimateNormals(xyz)
    xyz[77, 1] = 0.5
    nrm, _, _ = ctx.EstimateNormals(xyz)  # the context stays usable
    assert bool(torch.isfinite(nrm).all())
    ctx.close()
