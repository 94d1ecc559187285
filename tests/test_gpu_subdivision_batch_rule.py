"""Whether a batch bounds its subdivision tiles follows from the tiles of all its
clouds together (2048): two small clouds do without, and each mesh is the single
call's, index for index and bit for bit, on both sides of the line.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,depth,bounded", [([4000, 4000], 5, False), ([900] * 3, 6, None), ([5000] * 16, 6, True),
                                                 ([5000, 20000], 7, True)])
def test_batch(pkg, sizes, depth, bounded):
    import torch
    print("sizes", sizes, depth, flush=True)
    clouds = []
    for i, n in enumerate(sizes):
        x, m = pkg.synth.batch64(count=1, seed=100 + i, lo=n, hi=n)[0]
        clouds.append((torch.from_numpy(x).cuda(), torch.from_numpy(m).cuda()))
    batch = pkg.PoissonReconstruction(depth=depth, batch_cg_plan=0)
    meshes = batch.ReconstructBatch(clouds)
    L, tiles = pkg.binding.lib(), 0
    signs = pkg.binding.ARRAY_ID["SUBDIV_TILE_SIGNS"]
    for i in range(len(sizes)):
        need = ctypes.c_uint64(0)
        assert L.psr_export(L.psr_batch_cloud(batch._ctx, i), signs, None, 0, ctypes.byref(need)) == 0
        tiles += need.value // 4
    print("bounded tiles", tiles, flush=True)
    assert tiles == 0 or tiles >= 2048
    if bounded is not None:
        assert (tiles > 0) == bounded
    single = pkg.PoissonReconstruction(depth=depth)
    for i in (0, len(sizes) - 1):
        v, t = batch.mesh_to_host(meshes[i])
        single.SolvePoissionReconstructionMesh(*clouds[i])
        np.testing.assert_array_equal(t, single.GetRebuildMeshTriangleIndices())
        np.testing.assert_array_equal(v.view(np.int32), single.GetRebuildMeshVertices().view(np.int32))
    single.close()
    batch.close()
