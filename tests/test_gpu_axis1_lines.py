"""Grids whose axis 1 has no compiled kernel: an insertion's energies are its
own, bit for bit the same whatever insertions share its launch, and finite
beside one that is not."""
import numpy as np
import pytest

import erutil as U
from erdst_gpu import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ms", [
    (60, 30, 50),   # even length
    (45, 21, 35),   # odd length, an odd number of lines
    (60, 64, 64),   # under a compiled plane
    (420, 16, 18),  # the fewest lines per workgroup
])
def test_insertions_stay_apart(ms):
    w = synth.refs_water(0, 1000, 31.04, 19, 1, 32)
    w.params["ms"] = ms
    p = U.workload_params(w)
    ctx = capi.Context(w.topo, p)
    mesh, core = synth.linear_log_mesh(-80.0, 5.0, 0.17, 1.0e4, 100)
    ctx.set_mesh(np.array([len(mesh)], np.int32), np.array([len(mesh) - core], np.int32), mesh)
    ctx.set_solute(w.topo.slt_ljtype, w.topo.slt_charge32)
    ctx.set_frame(w.frame(0), w.cell)

    def energies(x):
        ctx.set_insertions(x)
        ctx.run(capi.ER_BATCHED)
        return ctx.uvengy()

    x = w.insertions(0).astype(np.float32)
    u, u0 = energies(x)
    assert np.isfinite(u).all()
    uo, _ = U.oracle_refs(w, 0, p)
    nbad, worst, at = U.energy_mismatch(u, uo, 5)
    assert nbad == 0, (worst, at, u[at], uo[at])
    moved, lost = x.copy(), x.copy()
    moved[::2] += np.float32(1.5)
    lost[::2] = np.nan
    for other in (moved, lost):
        v, _ = energies(other)
        np.testing.assert_array_equal(v[1::2], u[1::2])
    ctx.close()
