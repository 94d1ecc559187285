"""The subdivision's left-out tiles against every tile evaluated: the same cloud
with the bound forced on and forced off must give the same vertices and indices,
bit for bit, and the bound must have left tiles out, in roots of 8 to 64 cells a
side, alone in their set and in sets of several that touch.
"""
import os

import numpy as np
import pytest

from test_gpu_subdivision_bound import _cloud

pytestmark = pytest.mark.gpu


def _mesh(pkg, tx, tn, depth, tiles, **cfg):
    os.environ["PSR_SUBDIV_BOUND_TILES"] = str(tiles)
    try:
        rec = pkg.PoissonReconstruction(depth=depth, **cfg)
    finally:
        os.environ.pop("PSR_SUBDIV_BOUND_TILES")
    rec.SolvePoissionReconstructionMesh(tx, tn)
    out = rec.GetRebuildMeshVertices(), rec.GetRebuildMeshTriangleIndices(), rec.export("SUBDIV_TILE_SIGNS"), rec.stats()
    rec.close()
    return out


def _points(pkg, name):
    if name == "two":  # two scans far apart: large roots on both sides of the domain's middle
        a, b = pkg.synth.sphere(n=700, seed=3), pkg.synth.torus(n=900, seed=4)
        return np.concatenate([0.3 * a[0], 0.4 * b[0] + np.float32(0.6)]), np.concatenate([a[1], b[1]])
    if name == "few":
        return pkg.synth.displaced_sphere(n=2500)
    return _cloud(pkg, name)


@pytest.mark.parametrize("name,depth,prec", [("holes", 6, 1), ("holes", 7, 0), ("sparse", 5, 1), ("sparse", 7, 1), ("sparse", 8, 0),
                                             ("two", 7, 0), ("two", 6, 1), ("few", 8, 1), ("torus", 7, 1)])
def test_mesh_is_the_same_without_the_bound(pkg, name, depth, prec):
    import torch
    print("cloud", name, depth, prec, flush=True)
    xyz, nrm = _points(pkg, name)
    tx, tn = torch.from_numpy(np.ascontiguousarray(xyz)).cuda(), torch.from_numpy(np.ascontiguousarray(nrm)).cuda()
    v, t, none, _ = _mesh(pkg, tx, tn, depth, 1 << 30, precision=prec)
    w, u, signs, st = _mesh(pkg, tx, tn, depth, 0, precision=prec)
    print("q1", st["q1_fired"], "roots", st["roots"], "coarse", st["coarse_roots"], "tiles", len(signs), "left out",
          int((signs > 0).sum()), int((signs < 0).sum()), "triangles", len(t), flush=True)
    assert st["q1_fired"] == 0 and len(t) > 0
    assert len(none) == 0 and (signs != 0).any()
    np.testing.assert_array_equal(t, u)
    np.testing.assert_array_equal(v.view(np.int32), w.view(np.int32))
