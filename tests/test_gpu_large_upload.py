"""Host inputs beyond the 32 MiB that go through the page-locked ring: uploads
just below, at and above it give the energies of the same coordinates in
device memory, bit for bit, also right behind a run that still reads the
buffer."""
import numpy as np
import pytest
import torch

import erutil as U
from erdst_gpu import capi, synth
from erdst_gpu.topology import build_topology

pytestmark = pytest.mark.gpu
NSITE = 512
FULL = (32 << 20) // (NSITE * 12)  # insertions in 32 MiB, rounded down


@pytest.mark.parametrize("nins", [FULL, FULL + 1, FULL + 333])
def test_upload_sizes(nins):
    rng = np.random.default_rng(3)
    L = 31.04
    solute = synth.random_solute(rng, "s", NSITE)
    w = synth.refs_water(0, 24, L, 1, 1, 32)
    w.topo = build_topology([synth.water_species(24), solute], solute_index=1, refs=True)
    p = U.workload_params(w, cltype=0, corrcal=0)
    x = (rng.uniform(0.0, L, (nins, 1, 3)) + solute.geometry).astype(np.float32)
    y = np.ascontiguousarray(x[::-1])
    mesh, core = synth.linear_log_mesh(-400.0, 5.0, 5.0, 1.0e4, 10)
    ctx = capi.Context(w.topo, p)
    ctx.set_mesh(np.array([len(mesh)], np.int32), np.array([len(mesh) - core], np.int32), mesh)
    ctx.set_solute(w.topo.slt_ljtype, w.topo.slt_charge32)
    ctx.set_frame(w.frame(0), w.cell)
    ctx.set_insertions(y)
    ctx.run(capi.ER_BATCHED)
    ctx.set_insertions(x)  # the run above reads the same buffer
    u, _ = ctx.uvengy()
    ctx.run(capi.ER_BATCHED)
    v, _ = ctx.uvengy()
    np.testing.assert_array_equal(u, v[::-1])
    dev = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    ctx.set_insertions_device(nins, dev.data_ptr())
    ctx.run(capi.ER_BATCHED)
    np.testing.assert_array_equal(ctx.uvengy()[0], v)
    ctx.close()
