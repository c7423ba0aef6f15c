"""The frame's counting sorts at the sizes where they change form (one
workgroup up to 12288 molecules and atoms together, brick counters in LDS up
to 8192 bricks), against the FP64 oracle at the standing energy bar; and a
context of more solutes than a launch takes pointers for, against one context
per solute, bit for bit, over frames uploaded with no wait between."""
import numpy as np
import pytest

import erutil as U
from erdst_gpu import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,ms,order", [
    (3071, 48, 4), (3072, 48, 4), (3073, 48, 4),  # one workgroup, its last size, several
    (3000, 128, 6),                               # 16384 bricks: counters in memory
])
def test_frame_sorts(waters, ms, order):
    w = synth.refs_water(0, waters, 46.0, 3, 1, ms)
    p = U.workload_params(w, splodr=order)
    ctx = capi.Context(w.topo, p)
    mesh, core = synth.linear_log_mesh(-80.0, 5.0, 0.17, 1.0e4, 100)
    ctx.set_mesh(np.array([len(mesh)], np.int32), np.array([len(mesh) - core], np.int32), mesh)
    ctx.set_solute(w.topo.slt_ljtype, w.topo.slt_charge32)
    ctx.set_frame(w.frame(0), w.cell)
    ctx.set_insertions(w.insertions(0))
    ctx.run(capi.ER_BATCHED)
    ctx.sync()
    u, _ = ctx.uvengy()
    ctx.close()
    uo, _ = U.oracle_refs(w, 0, p)
    nbad, worst, at = U.energy_mismatch(u, uo, w.topo.slt_charge32.size)
    assert nbad == 0, (worst, at, u[at], uo[at])


@pytest.mark.parametrize("nsolute", [16, 17, 40])
def test_many_solutes(nsolute):
    w = synth.refs_water(0, 1000, 31.04, 5, 2, 32)
    p = U.workload_params(w)
    mesh, core = synth.linear_log_mesh(-80.0, 5.0, 0.17, 1.0e4, 100)
    mesh3 = (np.array([len(mesh)], np.int32), np.array([len(mesh) - core], np.int32), mesh)
    solute = (w.topo.slt_ljtype, w.topo.slt_charge32)

    def insertions(f, k):  # each solute its own count and places
        return np.roll(w.insertions(f), k, axis=1)[:1 + k % 5] if k % 2 else w.insertions(f)[:1 + k % 5]

    multi = capi.Context(w.topo, p)
    multi.set_mesh(*mesh3)
    multi.set_solutes([solute] * nsolute)
    for f in (0, 1):  # uploads follow the runs with no wait between
        multi.set_frame(w.frame(f), w.cell)
        for k in range(nsolute):
            multi.select_solute(k)
            multi.set_insertions(insertions(f, k))
        multi.run(capi.ER_BATCHED)
    for k in range(nsolute):
        single = capi.Context(w.topo, p)  # its own: the weights' offset outlives a clear
        single.set_mesh(*mesh3)
        single.set_solute(*solute)
        for f in (0, 1):
            single.set_frame(w.frame(f), w.cell)
            single.set_insertions(insertions(f, k))
            single.run(capi.ER_BATCHED)
        multi.select_solute(k)
        um, u0m = multi.uvengy()
        us, u0s = single.uvengy()
        np.testing.assert_array_equal(um, us)
        np.testing.assert_array_equal(u0m, u0s)
        gm, gs = multi.fetch(), single.fetch()
        np.testing.assert_array_equal(gm["edens"], gs["edens"])
        assert gm["engnorm"] == gs["engnorm"]
        single.close()
    multi.close()
