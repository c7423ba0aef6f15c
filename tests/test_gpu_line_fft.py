"""Grid lengths without a compiled plane or line kernel: the factored LDS
transforms (er_linefft.h) and, for prime factors above 7, the direct ones,
against the FP64 oracle at the standing energy bar (erutil.energy_tolerance)."""
import numpy as np
import pytest

import erutil as U
from erdst_gpu import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsite", [5, 12, 25])  # product form, its most sites, spread + transform
@pytest.mark.parametrize("ms,order", [
    ((16, 16, 18), 4),    # one factor per line and two
    ((45, 49, 42), 6),    # odd K1, factors 7 x 7 and 6 x 7
    ((98, 21, 50), 5),    # three factors along axis 1
    ((125, 28, 30), 4),   # 5 x 5 x 5, four lines per workgroup along axis 1
    ((256, 20, 75), 4),   # 16 x 16, one line of K2 K3 left over per group of lines
    ((64, 90, 105), 4),   # compiled axis 1 under a factored plane of 75 KB
    ((60, 64, 64), 4),    # factored axis 1 under a compiled plane
    ((62, 30, 33), 4),    # prime factors 31 and 11: both stages direct
])
def test_line_lengths(ms, order, nsite):
    solute = synth.tetra_species() if nsite == 5 else synth.random_solute(np.random.default_rng(nsite), "s", nsite)
    w = synth.refs_water(0, 1000, 31.04, 19, 1, 32, solute=solute)
    w.params["ms"] = ms
    p = U.workload_params(w, splodr=order)
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
