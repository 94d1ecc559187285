"""Batches of few clouds under every CG plan: a plan of several waves of the
resident budget must not ask more workgroups of one cloud than can be resident
(such calls failed with "CG launch exceeds the resident workgroup budget", the
tuner's trials of them among the first calls of a default batch).

Each solution's residual is recomputed on the host in FP64, with the bounds of the
single call: 1e-4 of ||b|| in the FP32 form, 1e-5 and a margin of 1e-6 in the mixed.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")  # before the library: both share one HIP runtime

pytestmark = pytest.mark.gpu


def _up(cloud):
    return tuple(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in cloud)


def _check(batch, i, depth, prec):
    import residual_host
    rel = residual_host.true_relres(batch.batch_cloud(i), depth)
    st = batch.batch_stats(i)
    print("cloud", i, "workgroups", st["cg_workgroups"], "row form", st["cg_row_form"], "relres", max(rel), flush=True)
    assert st["q1_fired"] == 0
    assert max(rel) <= (1e-4 if prec == 0 else 1e-5 + 1e-6)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("plan", [1, 2, 4, 8])
def test_plan(pkg, plan, prec):
    print("plan", plan, prec, flush=True)
    batch = pkg.PoissonReconstruction(depth=7, precision=prec, batch_cg_plan=plan)
    meshes = batch.ReconstructBatch([_up(pkg.synth.torus(n=200000)), _up(pkg.synth.sphere(n=20000))])
    assert batch.batch_cg_plan() == plan and all(m.n_triangles > 0 for m in meshes)
    _check(batch, 0, 7, prec)
    _check(batch, 1, 7, prec)
    batch.close()


@pytest.mark.parametrize("prec", [0, 1])
def test_tuner_tries_every_plan(pkg, prec):
    """The first call and a trial of each of the five plans, then the one it keeps."""
    print("precision", prec, flush=True)
    cloud = _up(pkg.synth.torus(n=150000, seed=5))
    batch = pkg.PoissonReconstruction(depth=7, precision=prec)
    plans = []
    for _ in range(8):
        assert batch.ReconstructBatch([cloud])[0].n_triangles > 0
        plans.append(batch.batch_cg_plan())
    print("plans", plans, flush=True)
    assert plans[1:6] == [0, 1, 2, 4, 8] and plans[6] == plans[7]
    _check(batch, 0, 7, prec)
    batch.close()


def test_plan_at_an_indefinite_depth(pkg):
    """Depth 9 in the mixed form: the MINRES launch has a budget of its own."""
    xyz, nrm = pkg.synth.batch64(count=1, seed=7, lo=40000, hi=40000)[0]
    batch = pkg.PoissonReconstruction(depth=9, precision=1, batch_cg_plan=8, cg_max_iter=300)
    assert batch.ReconstructBatch([_up((xyz, nrm))])[0].n_triangles > 0
    rep = batch.batch_stats(0)["cg_true_relres"]
    import residual_host
    host = residual_host.true_relres(batch.batch_cloud(0), 9)
    print("reported", rep, "host", host, flush=True)
    assert np.all(np.abs(np.array(host) - rep) <= 1e-3 * np.maximum(rep, 1e-6))
    batch.close()
