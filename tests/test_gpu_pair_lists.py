"""The pair searches where one workgroup meets more molecules than its list
holds (2048): the energies are the same, bit for bit, whatever the split and
from run to run, and those of the FP64 oracle.  Bare Coulomb, as in
test_gpu_pairs_many; the solute is a straight chain, so long or with so long a
cutoff that the search holds 2300 to 2800 molecules (or, over 4096, three lists)."""
import numpy as np
import pytest

import erutil as U
from erdst_gpu import capi, synth
from erdst_gpu.topology import Species, build_topology

pytestmark = pytest.mark.gpu
L, NWATER, NCHAIN, CHAIN, NINS = 62.0, 6200, 900, 17, 3


def _workload(nsite):
    rng = np.random.default_rng(nsite)
    q = rng.normal(0.0, 0.2, CHAIN)
    sp = Species("chain", NCHAIN, q - q.mean(), rng.uniform(0.03, 0.2, CHAIN), rng.uniform(3.0, 4.0, CHAIN),
                 synth.random_chain(rng, CHAIN))
    q = rng.normal(0.0, 0.3, nsite)
    rod = np.stack([1.2 * np.arange(nsite), np.zeros(nsite), np.zeros(nsite)], 1)
    solute = Species("rod", 1, q - q.mean(), rng.uniform(0.03, 0.2, nsite), rng.uniform(2.5, 3.5, nsite),
                     rod - rod.mean(0))
    w = synth.refs_water(0, 1000, L, NINS, 1, 64)
    w.topo = build_topology([sp, synth.water_species(NWATER), solute], solute_index=2, refs=True)
    c = synth.lattice_centres(rng, NCHAIN + NWATER, np.array([L] * 3))
    pos = np.concatenate([synth.place_rigid(rng, sp.geometry, c[:NCHAIN]),
                          synth.place_rigid(rng, synth.water_geometry(), c[NCHAIN:])]).astype(np.float32)
    ins = synth.place_rigid(rng, solute.geometry, rng.uniform(0.0, L, (NINS, 3)))
    w._frame_fn = lambda f: pos
    w._ins_fn = lambda f: ins.reshape(NINS, nsite, 3).astype(np.float32)
    mesh, core = synth.linear_log_mesh(-400.0, 5.0, 0.81, 1.0e4, 100)
    w.mesh = [(mesh, core)] * 2
    return w


def _in_sphere(w, cut):
    """Per insertion: molecules with an atom nearer to the solute's centre than
    the cutoff and its reach (the search lists every one of them)."""
    t, pos = w.topo, w.frame(0).astype(np.float64)
    out = []
    for x in w.insertions(0).astype(np.float64):
        c = x.mean(0)
        d = pos - c
        d -= L * np.round(d / L)
        near = np.sqrt((d * d).sum(-1)) < cut + np.sqrt(((x - c) ** 2).sum(-1)).max()
        out.append(int(np.logical_or.reduceat(near, t.mol_begin[:-1]).sum()))
    return out


def _at_cutoff(w, cut):
    """[insertions, molecules]: a site pair within 2e-7 of the cutoff, relative (a few
    roundings of an FP32 distance)."""
    t, pos = w.topo, w.frame(0).astype(np.float64)
    out = np.zeros((w.nins, t.nmol), bool)
    for n, x in enumerate(w.insertions(0).astype(np.float64)):
        edge = np.zeros(len(pos), bool)
        for s in x:
            d = s - pos
            d -= L * np.round(d / L)
            edge |= np.abs(np.sqrt((d * d).sum(-1)) - cut) < 2e-7 * cut
        out[n] = np.logical_or.reduceat(edge, t.mol_begin[:-1])
    return out


@pytest.mark.parametrize("nsite,cut,least", [(25, 12.0, 2048), (9, 29.0, 4096), (5, 26.0, 2048)])
def test_full_candidate_list(nsite, cut, least):
    w = _workload(nsite)
    assert min(_in_sphere(w, cut)) > least  # in one part with a split of 1
    p = U.workload_params(w, cltype=0, elecut=cut, upljcut=cut, lwljcut=cut - 2.0)
    first = None
    for split in (64, 1, 1, 1, 2, 0):
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
            uo, _ = U.oracle_refs(w, 0, p)
            edge = _at_cutoff(w, cut)
            assert edge.sum() <= 9
            nbad, worst, at = U.energy_mismatch(np.where(edge, uo, u), uo, nsite)
            assert nbad == 0, (worst, at, u[at], uo[at])
        assert np.array_equal(u, first), (split, int((u != first).sum()))
