"""The compiled plane kernels at each thread count of the dispatch (256, 512,
768 and the planes that fill a CU), product and spread forms, one and two
chunks of site factors, against the FP64 oracle at the standing energy bar
(erutil.energy_tolerance)."""
import numpy as np
import pytest

import erutil as U
from erdst_gpu import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsite", [5, 9, 20])
@pytest.mark.parametrize("k", [48, 64, 80, 96, 108])
def test_plane_threads(k, nsite):
    solute = synth.tetra_species() if nsite == 5 else synth.random_solute(np.random.default_rng(nsite), "s", nsite)
    w = synth.refs_water(0, 1000, 31.04, 3, 1, 32, solute=solute)
    w.params["ms"] = (32, k, k)
    p = U.workload_params(w, splodr=4)
    ctx = capi.Context(w.topo, p)
    mesh, core = synth.linear_log_mesh(-80.0, 5.0, 0.17, 1.0e4, 100)
    ctx.set_mesh(np.array([len(mesh)], np.int32), np.array([len(mesh) - core], np.int32), mesh)
    ctx.set_solute(w.topo.slt_ljtype, w.topo.slt_charge32)
    ctx.set_frame(w.frame(0), w.cell)
    ctx.set_insertions(w.insertions(0))
    ctx.run(capi.ER_BATCHED)
    ctx.sync()
    u, u0 = ctx.uvengy()
    ctx.close()
    uo, u0o = U.oracle_refs(w, 0, p)
    nbad, worst, at = U.energy_mismatch(u, uo, nsite)
    assert nbad == 0, (worst, at, u[at], uo[at])
    assert U.self_mismatch(u0, u0o, nsite)[0] == 0
