"""Which form of the solver runs is reported depth by depth (CG_FORM), and the
forms that must agree do: the MINRES with its vectors on chip makes the same
operations in the same order as the one in memory at the same row blocks, so
solution, iterations and mesh are equal to the bit; clouds and row blocks meant
for the one-row form run it.
"""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # before the library: both share one HIP runtime

pytestmark = pytest.mark.gpu


def _run(pkg, cloud, depth, prec, env, **cfg):
    os.environ.update(env)
    try:
        rec = pkg.PoissonReconstruction(depth=depth, precision=prec, **cfg)
    finally:
        for k in env:
            del os.environ[k]
    rec.SolvePoissionReconstructionMesh(*(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in cloud))
    return rec


@pytest.mark.parametrize("rows,n,form", [(None, 3000, 4), (1024, 6000, 4), (1032, 3000, 8), (2048, 6000, 8), (4096, 6000, 16),
                                         (4096, 500, 16), (300, 3000, 4)])
def test_minres_on_chip_equals_memory(pkg, rows, n, form):
    print("rows", rows, "points", n, flush=True)
    cloud = pkg.synth.batch64(count=1, seed=7, lo=n, hi=n)[0]
    env = {"PSR_CG_ROWS_PER_WG": str(rows)} if rows else {}
    got = []
    for memory in (False, True):
        rec = _run(pkg, cloud, 9, 1, {**env, "PSR_CG_MINRES_IN_MEMORY": "1"} if memory else env, cg_max_iter=400)
        forms, st = rec.export("CG_FORM"), rec.stats()
        print("forms", forms, "iterations", st["cg_iterations"], "relres", st["cg_true_relres"][9], flush=True)
        assert forms[9] == (-1 if memory else form)
        got.append((rec.export("DX"), np.array(st["cg_iterations"]), rec.GetRebuildMeshVertices(), rec.GetRebuildMeshTriangleIndices()))
        rec.close()
    for a, b in zip(*got):
        assert a.shape == b.shape and np.array_equal(a.view(np.int32), b.view(np.int32))


def test_rows_beyond_the_registers_go_to_memory(pkg):
    rec = _run(pkg, pkg.synth.batch64(count=1, seed=7, lo=6000, hi=6000)[0], 9, 1, {"PSR_CG_ROWS_PER_WG": "8192"}, cg_max_iter=50)
    forms = rec.export("CG_FORM")
    rec.close()
    assert forms[9] == -1


def _volume(n, seed):
    r = np.random.RandomState(seed)
    nrm = r.standard_normal((n, 3))
    return r.rand(n, 3).astype(np.float32), (nrm / np.linalg.norm(nrm, axis=1, keepdims=True)).astype(np.float32)


@pytest.mark.parametrize("rows", [None, 8, 100, 256])
@pytest.mark.parametrize("cloud,depth", [("sphere", 5), ("volume", 5), ("volume", 6), ("pair", 3)])
@pytest.mark.parametrize("prec", [0, 1])
def test_one_row_form_runs_where_it_fits(pkg, rows, cloud, depth, prec):
    """The clouds and row blocks whose residuals test_gpu_cg_rows checks: a row per thread wherever all workgroups are
    resident, four a CU in the FP32 form and three in the mixed, several rows beyond (8 rows a workgroup)."""
    print("rows", rows, cloud, depth, prec, flush=True)
    c = {"sphere": lambda: pkg.synth.sphere(n=4000), "volume": lambda: _volume(3000 if depth == 5 else 8000, depth),
         "pair": lambda: pkg.synth.sphere(n=64)}[cloud]()
    rec = _run(pkg, c, depth, prec, {"PSR_CG_ROWS_PER_WG": str(rows)} if rows else {}, cg_max_iter=3)
    forms, counts = rec.export("CG_FORM"), rec.export("LEVEL_COUNT").astype(int)
    rec.close()
    workgroups = int((-(-counts // (rows or 512))).sum())
    resident = (4 if prec == 0 else 3) * torch.cuda.get_device_properties(0).multi_processor_count
    print("workgroups", workgroups, "of", resident, "forms", forms, flush=True)
    assert np.all(forms == (1 if workgroups <= resident else 0))
    assert rows == 8 or workgroups <= resident
