"""The neighbours' d_x copied four entries a thread, at node counts whose 27-fold
leaves every remainder, on the regular grid and on bent neighbour tables: seen
through the implicit function at the points, whose every term reads one.

The host sums the same float products in FP64 over a point's leaf and ancestors;
the device in float: at most 27 (depth + 1) terms, each of relative error 8 2^-24
with its sum's, so 300 2^-24 of the terms' sum of magnitudes is asked.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spline(u):
    u = np.abs(u)
    return np.where(u < 0.5, 1 - 4 / 3 * u * u, np.where(u < 1.5, 2 / 3 * (1.5 - u) ** 2, 0.0))


@pytest.mark.parametrize("cloud,depth", [("sphere", 2), ("sphere", 3), ("sphere", 4), ("sphere", 6), ("bent", 7)])
def test_point_values(pkg, cloud, depth):
    import torch
    xyz, nrm = pkg.synth.batch64()[36] if cloud == "bent" else pkg.synth.sphere(n=900)
    rec = pkg.PoissonReconstruction(depth=depth, precision=1)
    rec.SolvePoissionReconstructionMesh(torch.from_numpy(xyz).cuda(), torch.from_numpy(nrm).cuda())
    base = rec.export("LEVEL_BASE").astype(np.int64)
    enc = rec.export("NODE_ENCIDX").reshape(-1).astype(np.int64)
    neigh = rec.export("NODE_NEIGHS").reshape(-1, 27).astype(np.int64)
    parent = rec.export("NODE_PARENT").reshape(-1).astype(np.int64)
    dx, chi = rec.export("DX").astype(np.float64), rec.export("CHI_POINTS").astype(np.float64)
    pos = rec.export("SORTED_POS")[:, :3].astype(np.float64)
    now = base[depth] + rec.export("POINT2NODE").reshape(-1).astype(np.int64)
    print(cloud, depth, "nodes", len(enc), "q1", rec.stats()["q1_fired"], flush=True)
    rec.close()
    s1 = 1 << (depth + 1)
    f = np.stack([enc & (s1 - 1), (enc >> (depth + 1)) & (s1 - 1), enc >> (2 * (depth + 1))], 1)
    lev = np.floor(np.log2(f + 1)).astype(np.int64)
    centre, inv = (f + 1 - (1 << lev) + 0.5) / (1 << lev), (1 << lev).astype(np.float64)
    want, mag = np.zeros(len(pos)), np.zeros(len(pos))
    while (now >= 0).any():
        for q in range(27):
            nb = np.where(now >= 0, neigh[now, q], -1)
            ok = nb >= 0
            term = dx[nb] * np.prod(_spline((pos - centre[nb]) * inv[nb]), 1)
            want += np.where(ok, term, 0)
            mag += np.where(ok, np.abs(term), 0)
        now = np.where(now >= 0, parent[now], -1)
    assert np.all(np.abs(chi - want) <= 300 * 2.0**-24 * mag + 1e-30)
