"""The stored operator against the one rebuilt on the host from the 1-D tables:
on the regular grid (an entry is its depth's and offset's constant) and on a
cloud whose neighbour tables the child 0 rule bends (an entry per pair of
nodes).

The kept entries per depth are whole numbers and must be equal.  The entries'
values show in the mixed form's reported residual, which the solver takes with
its own entries and the host with the rebuilt ones: both are FP64 sums of the
same floats, asked to agree to 1e-3 of the larger of themselves and 1e-6.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _kept(rec, D):
    import residual_host
    res = (1 << (D + 1)) - 1
    dot, d2 = (rec.export(k).reshape(res, res) for k in ("TABLE_DOT", "TABLE_D2DOT"))
    f = residual_host.decode(rec.export("NODE_ENCIDX").astype(np.int64).reshape(-1), D)
    neigh = rec.export("NODE_NEIGHS").reshape(-1, 27)
    base = rec.export("LEVEL_BASE").astype(np.int64)
    o, q = np.nonzero(neigh >= 0)
    j = neigh[o, q]
    s = [(a[o], a[j]) for a in f]
    e = dot[s[0]] * dot[s[1]] * dot[s[2]] * (d2[s[0]] + d2[s[1]] + d2[s[2]])
    rows = o[np.abs(e) > float(np.float32(1e-6))]
    return [int(((rows >= base[d]) & (rows < base[d + 1])).sum()) for d in range(D + 1)]


@pytest.mark.parametrize("cloud,depth", [("sphere", 2), ("bent", 7), ("sphere", 5), ("torus", 7), ("torus", 8)])
def test_entries(pkg, cloud, depth):
    import residual_host
    import torch
    if cloud == "bent":
        xyz, nrm = pkg.synth.batch64()[36]
    else:
        xyz, nrm = pkg.synth.torus(n=60000) if cloud == "torus" else pkg.synth.sphere(n=4000)
    rec = pkg.PoissonReconstruction(depth=depth, precision=1)
    rec.SolvePoissionReconstructionMesh(torch.from_numpy(xyz).cuda(), torch.from_numpy(nrm).cuda())
    st, kept, rel = rec.stats(), _kept(rec, depth), residual_host.true_relres(rec, depth)
    rec.close()
    print(cloud, depth, "q1", st["q1_fired"], "kept", kept, "relres", rel, flush=True)
    assert st["q1_fired"] == (cloud == "bent")
    assert list(st["cg_nnz"])[:depth + 1] == kept
    rep = np.array(st["cg_true_relres"])[:depth + 1]
    assert np.all(np.abs(rep - rel) <= 1e-3 * np.maximum(rep, 1e-6))
