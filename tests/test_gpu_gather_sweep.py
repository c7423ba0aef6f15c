"""The sweeping order-6 gather (launches of four brick columns per CU or more)
at its edges: columns of an odd number of bricks and a half last brick, a step
with more atoms than its staged records, empty columns, a last tile of one
insertion, against the FP64 oracle at the standing energy bar
(erutil.energy_tolerance)."""
import numpy as np
import pytest

import erutil as U
from erdst_gpu import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ms", [(64, 60, 42), (60, 64, 45), (105, 90, 16)])
@pytest.mark.parametrize("layout", ["uniform", "cluster"])
def test_gather_sweep(ms, layout):
    L = 31.04
    nbx, nby = -(-ms[0] // 8), -(-ms[1] // 8)
    nins = 16 * -(-4 * 256 // (nbx * nby)) + 1  # one tile past four columns on each of 256 CUs
    w = synth.refs_water(0, 600, L, nins, 1, 32)
    w.params["ms"] = ms
    pos = w.frame(0).copy()
    if layout == "cluster":  # all in one corner: 300 in one brick's 2 A, the others in the lowest sixth
        rng = np.random.default_rng(7)
        c = np.concatenate([rng.uniform(1.2, 2.2, (300, 3)), rng.uniform(0.0, L / 6, (300, 3))])
        pos = synth.place_rigid(rng, synth.water_geometry(), c).astype(np.float32).reshape(pos.shape)
    w._frame_fn = lambda f: pos
    p = U.workload_params(w, splodr=6)
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
