"""Welding at the edges of its scan over workgroups and of its sort (a mesh of
few vertices, of one workgroup, of many; every depth's key length), and one
context welding meshes of different sizes in turn.

The welded mesh is whole numbers and copies: equal, bit for bit, to the numpy
restatement (first vertex of each key, ascending keys, corners through the
inverse map).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,sizes", [(2, [64]), (3, [300, 64]), (5, [4000, 64, 4000]), (7, [60000]), (8, [20000])])
def test_weld(pkg, depth, sizes):
    import torch
    rec = pkg.PoissonReconstruction(depth=depth, precision=1)
    for n in sizes:
        xyz, nrm = pkg.synth.sphere(n=n)
        rec.SolvePoissionReconstructionMesh(torch.from_numpy(xyz).cuda(), torch.from_numpy(nrm).cuda())
        v, t, key = rec.export("MESH_VERTICES"), rec.export("MESH_TRIANGLES"), rec.export("MESH_VERTEX_KEYS")
        wv, wt = rec.mesh_to_host(rec.WeldMesh())
        print("depth", depth, "points", n, "vertices", len(v), "welded", len(wv), flush=True)
        assert int(key.max()) < 3 * (2**depth + 1)**3
        _, first, inverse = np.unique(key, return_index=True, return_inverse=True)
        np.testing.assert_array_equal(wv.view(np.int32), v[first].view(np.int32))
        tt = t.reshape(-1, 3)
        ok = (tt >= 0) & (tt < len(v))
        want = np.where(ok, inverse.reshape(-1)[np.where(ok, tt, 0)], -1)
        np.testing.assert_array_equal(wt, want)
    rec.close()
