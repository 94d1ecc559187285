"""The MINRES of an indefinite depth with its vectors on chip: every number of
rows a thread holds, one workgroup and many, a last workgroup that is partly
empty, and the two ways out of it (row blocks that cut sibling blocks, so that
neighbours are read from memory; row blocks too long for the registers).

The reported FP64 residual must be that of the returned solution, recomputed on
the host from the exported operator: both are FP64 sums of the same float
values, so they agree to far better than the 1e-3 asked for.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reconstruct(pkg, rows, n):
    import torch
    xyz, nrm = pkg.synth.batch64(count=1, seed=7, lo=n, hi=n)[0]
    if rows:
        os.environ["PSR_CG_ROWS_PER_WG"] = str(rows)
    try:
        rec = pkg.PoissonReconstruction(depth=9, precision=pkg.binding.PRECISION_MIXED, cg_max_iter=600)
    finally:
        os.environ.pop("PSR_CG_ROWS_PER_WG", None)
    mesh = rec.SolvePoissionReconstructionMesh(torch.from_numpy(xyz).cuda(), torch.from_numpy(nrm).cuda())
    assert mesh.n_triangles > 0
    return rec


@pytest.mark.parametrize("rows,n", [(None, 3000), (256, 6000), (300, 3000), (1024, 6000), (1032, 3000), (2048, 6000),
                                    (4096, 6000), (4096, 500), (8192, 6000)])
def test_reported_residual_is_the_solutions(pkg, rows, n):
    import residual_host
    print("rows", rows, "points", n, flush=True)
    rec = _reconstruct(pkg, rows, n)
    st = rec.stats()
    rep, host = st["cg_true_relres"], residual_host.true_relres(rec, 9)
    print("iterations", st["cg_iterations"], "reported", rep[9], "host", host[9], flush=True)
    rec.close()
    assert 0 < st["cg_iterations"][9] <= 600
    assert np.isfinite(rep[9]) and rep[9] < 1.0
    assert abs(host[9] - rep[9]) <= 1e-3 * max(rep[9], 1e-6)


def test_barrier_time_out_is_reported(pkg):
    """A bound of zero polls ends every workgroup of the launch and fails the call; a context with the default bound works."""
    os.environ["PSR_CG_SPIN_LIMIT"] = "0"
    try:
        with pytest.raises(pkg.binding.PsrError, match="CG group barrier timed out"):
            _reconstruct(pkg, 256, 6000)
    finally:
        os.environ.pop("PSR_CG_SPIN_LIMIT", None)
    _reconstruct(pkg, 256, 6000).close()
