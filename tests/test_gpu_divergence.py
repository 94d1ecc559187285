"""The divergence against its definition on the host, in FP64, from the exported
vector field, tables and neighbours: every role of the launch (depths 0 to 3
shared out over workgroups, a wave per node between, a thread per node at depth
D) at the smallest and at a large depth, both field formats, on the regular grid
and on a cloud whose neighbour tables the child 0 rule bends.

Both are FP64 sums of the same products, the device's rounded to float at the
end: 2^-24 of the value, and 1e-10 of the depth's largest value for sums that
cancel (their terms' rounding, 1e-16 times at most 1e6 terms).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _divergence(rec, D):
    res = (1 << (D + 1)) - 1
    ddot = rec.export("TABLE_DDOT").reshape(res, res).T  # [a, b]: <F_a', F_b> is at a + res b
    enc = rec.export("NODE_ENCIDX").reshape(-1).astype(np.int64)
    s1 = 1 << (D + 1)
    f = np.stack([enc & (s1 - 1), (enc >> (D + 1)) & (s1 - 1), enc >> (2 * (D + 1))])
    neigh = rec.export("NODE_NEIGHS").reshape(-1, 27).astype(np.int64)
    didx, dnum = (rec.export(k).reshape(-1).astype(np.int64) for k in ("NODE_DIDX", "NODE_DNUM"))
    base = rec.export("LEVEL_BASE").astype(np.int64)
    v = rec.export("VFIELD").astype(np.float64)
    out = np.zeros(len(enc))
    for q in range(27):
        o = np.nonzero(neigh[:, q] >= 0)[0]
        nb = neigh[o, q]
        leaf = o >= base[D]
        first = np.where(leaf, nb - base[D], didx[nb])
        count = np.where(leaf, 1, dnum[nb])
        rows = np.repeat(o, count)
        j = np.repeat(first, count) + np.arange(count.sum()) - np.repeat(np.cumsum(count) - count, count)
        term = sum(v[j, a] * ddot[f[a][rows], f[a][base[D] + j]] for a in range(3))
        out += np.bincount(rows, term, len(enc))
    return out, base


@pytest.mark.parametrize("cloud,depth", [("sphere", 2), ("sphere", 4), ("sphere", 5), ("torus", 7), ("sphere", 8),
                                         ("bent", 7)])
@pytest.mark.parametrize("prec", [0, 1])
def test_divergence(pkg, cloud, depth, prec):
    import torch
    if cloud == "bent":
        xyz, nrm = pkg.synth.batch64()[36]
    else:
        xyz, nrm = pkg.synth.torus(n=20000) if cloud == "torus" else pkg.synth.sphere(n=1500)
    print(cloud, depth, prec, flush=True)
    rec = pkg.PoissonReconstruction(depth=depth, precision=prec)
    rec.SolvePoissionReconstructionMesh(torch.from_numpy(xyz).cuda(), torch.from_numpy(nrm).cuda())
    got = rec.export("DIVERGENCE").astype(np.float64)
    want, base = _divergence(rec, depth)
    rec.close()
    for d in range(depth + 1):
        a, b = got[base[d]:base[d + 1]], want[base[d]:base[d + 1]]
        assert np.all(np.abs(a - b) <= 2.0**-24 * 1.01 * np.abs(b) + 1e-10 * np.abs(b).max()), d
