"""Order 6 takes one of two gather kernels by the size of the launch
(k_gather_sweep from four brick columns per CU): the energies of an insertion
are the same, bit for bit, in chunks on either side of that line."""
import numpy as np
import pytest
import torch

import erutil as U
from erdst_gpu import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ms", [(64, 64, 64), (64, 60, 42)])
def test_chunks_agree(ms):
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = -(-4 * ncu // (-(-ms[0] // 8) * -(-ms[1] // 8)))  # the fewest of a sweep
    w = synth.refs_water(0, 1000, 31.04, 16 * tiles + 5, 1, 32)
    w.params["ms"] = ms
    p = U.workload_params(w, splodr=6)
    mesh, core = synth.linear_log_mesh(-80.0, 5.0, 0.17, 1.0e4, 100)
    out = []
    for chunk in (16 * (tiles + 1), 16 * tiles, 16 * (tiles - 1), 16):
        ctx = capi.Context(w.topo, p)
        ctx.set_mesh(np.array([len(mesh)], np.int32), np.array([len(mesh) - core], np.int32), mesh)
        ctx.set_solute(w.topo.slt_ljtype, w.topo.slt_charge32)
        ctx.set_tuning(dict(chunk=chunk, hist_slices=0, pair_split=[0], cell_width=0.0))
        ctx.set_frame(w.frame(0), w.cell)
        ctx.set_insertions(w.insertions(0))
        ctx.run(capi.ER_BATCHED)
        out.append(ctx.uvengy()[0])
        ctx.close()
    uo, _ = U.oracle_refs(w, 0, p, nins=16)
    nbad, worst, at = U.energy_mismatch(out[0][:16], uo, 5)
    assert nbad == 0, (worst, at, out[0][at], uo[at])
    for u in out[1:]:
        np.testing.assert_array_equal(u, out[0])
