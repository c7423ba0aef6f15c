"""The many-site pair search (k_pairs_many) at the edges of its work split:
site counts around the lane classes and the LDS share, molecules below, at
and above the segment threshold, against the FP64 oracle with bare Coulomb,
and the same energies bit for bit under every pair split.  Bare Coulomb stops
at the cutoff with a jump of several kcal/mol, so a molecule with a site pair
within 1e-6 A of it (FP32 rounding of a 12 A distance) has no energy to compare."""
import numpy as np
import pytest

import erutil as U
from erdst_gpu import capi, synth
from erdst_gpu.topology import Species, build_topology

pytestmark = pytest.mark.gpu


def _workload(nsite, chain, nins=5):
    """Water and a `chain`-site rigid chain in a 34 A cube, a random solute."""
    rng = np.random.default_rng(100 * nsite + chain)
    q = rng.normal(0.0, 0.2, chain)
    sp = Species("chain", 150, q - q.mean(), rng.uniform(0.03, 0.2, chain), rng.uniform(3.0, 4.0, chain),
                 synth.random_chain(rng, chain))
    solute = synth.random_solute(rng, "s", nsite)
    box = np.array([34.0] * 3)
    solvent = [sp, synth.water_species(700)]
    w = synth.refs_water(0, 1000, 34.0, nins, 1, 32)
    w.topo = build_topology(solvent + [solute], solute_index=2, refs=True)
    c = synth.lattice_centres(rng, 850, box)
    pos = np.concatenate([synth.place_rigid(rng, sp.geometry, c[:150]),
                          synth.place_rigid(rng, synth.water_geometry(), c[150:])]).astype(np.float32)
    ins = synth.place_rigid(rng, solute.geometry, rng.uniform(0.0, 34.0, (nins, 3)))
    w._frame_fn = lambda f: pos
    w._ins_fn = lambda f: ins.reshape(nins, nsite, 3).astype(np.float32)
    mesh, core = synth.linear_log_mesh(-400.0, 5.0, 0.81, 1.0e4, 100)
    w.mesh = [(mesh, core)] * 2
    return w


def _at_cutoff(w):
    """[insertions, molecules]: a site pair within 1e-6 A of the 12 A cutoff."""
    t, pos = w.topo, w.frame(0).astype(np.float64)
    out = np.zeros((w.nins, t.nmol), bool)
    for n, x in enumerate(w.insertions(0).astype(np.float64)):
        d = x[:, None, :] - pos[None, :, :]
        d -= 34.0 * np.round(d / 34.0)
        edge = (np.abs(np.sqrt((d * d).sum(-1)) - 12.0) < 1e-6).any(0)
        out[n] = np.logical_or.reduceat(edge, t.mol_begin[:-1])
    return out


@pytest.mark.parametrize("nsite", [9, 16, 17, 33, 64, 65, 150, 256, 257, 600])
@pytest.mark.parametrize("chain", [5, 16, 17, 41])
def test_pairs_many(nsite, chain):
    w = _workload(nsite, chain)
    p = U.workload_params(w, cltype=0)
    uo, _ = U.oracle_refs(w, 0, p)
    edge = _at_cutoff(w)
    assert edge.sum() <= 2
    first = None
    for split in (0, 1, 7, 64):
        ctx = capi.Context(w.topo, p)
        ctx.set_mesh(*w.uvmax_uvsoft_uvcrd())
        ctx.set_solute(w.topo.slt_ljtype, w.topo.slt_charge32)
        ctx.set_tuning(dict(chunk=0, hist_slices=0, pair_split=[split], cell_width=0.0))
        ctx.set_frame(w.frame(0), w.cell)
        ctx.set_insertions(w.insertions(0))
        ctx.run(capi.ER_BATCHED)
        u, _ = ctx.uvengy()
        ctx.close()
        if first is None:
            first = u
            nbad, worst, at = U.energy_mismatch(np.where(edge, uo, u), uo, nsite)
            assert nbad == 0, (worst, at, u[at], uo[at])
        assert np.array_equal(u, first), split
