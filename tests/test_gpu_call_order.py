"""Calls between runs: what er_get_flceng gives after the solute list grows,
a context after a call that it refused, inputs where the kernels cannot reach
them."""
import ctypes

import numpy as np
import pytest
import torch

import erutil as U
from erdst_gpu import capi, synth

pytestmark = pytest.mark.gpu


def test_flceng_outlives_a_longer_solute_list():
    """er_get_flceng gives the last run's sums until the next run, also after
    er_set_solute_molecules has named more molecules than that run had."""
    w = synth.soln_water(0, 1000, 31.04, 1, 32)
    ctx = capi.Context(w.topo, U.workload_params(w))
    ctx.set_mesh(*w.uvmax_uvsoft_uvcrd())
    ctx.set_solute_molecules([1, 2])  # two of the waters
    ctx.set_frame(w.frame(0), w.cell)
    ctx.run(capi.ER_BATCHED)
    before = ctx.flceng(2)
    assert np.all(before != 0.0)
    ctx.set_solute_molecules(np.arange(1, 901))
    np.testing.assert_array_equal(ctx.flceng(2), before)
    ctx.run(capi.ER_BATCHED)
    np.testing.assert_allclose(ctx.flceng(900)[:2], before, rtol=1e-6)
    ctx.close()


def _refs_ctx(w, solutes):
    ctx = capi.Context(w.topo, U.workload_params(w))
    ctx.set_mesh(*w.uvmax_uvsoft_uvcrd())
    ctx.set_solutes(solutes)
    return ctx


def _run(ctx, w, nsolute, nins=5):
    ctx.set_frame(w.frame(0), w.cell)
    for k in range(nsolute):
        ctx.select_solute(k)
        ctx.set_insertions(w.insertions(0)[k:k + nins])
    ctx.run(capi.ER_BATCHED)
    ctx.sync()
    out = []
    for k in range(nsolute):
        ctx.select_solute(k)
        out.append((ctx.uvengy(), ctx.fetch()))
    return out


@pytest.mark.parametrize("before,refused", [(1, 2), (1, 40), (3, 2)])
def test_refused_solutes_change_nothing(before, refused):
    """er_set_solutes with a bad last solute: no halt out of nowhere, and the
    context runs, clears and fetches as if the call had not been made."""
    w = synth.refs_water(0, 1000, 31.04, 8, 1, 32)
    good = (w.topo.slt_ljtype, w.topo.slt_charge32)
    bad = (np.full(5, w.topo.ntype), w.topo.slt_charge32)  # 0-based: one past the types
    want = _refs_ctx(w, [good] * before)
    ctx = _refs_ctx(w, [good] * before)
    with pytest.raises(capi.ErError) as ei:
        ctx.set_solutes([good] * (refused - 1) + [bad])
    assert ei.value.status == capi.ER_E_ARG
    ctx.sync()
    ctx.clear()
    for (ua, ga), (ub, gb) in zip(_run(ctx, w, before), _run(want, w, before), strict=True):
        np.testing.assert_array_equal(ua[0], ub[0])
        np.testing.assert_array_equal(ga["edens"], gb["edens"])
        assert ga["engnorm"] == gb["engnorm"]
    ctx.close()
    want.close()


def test_refused_mesh_changes_nothing():
    """er_set_mesh with a longer mesh that does not increase: the context
    clears, runs and fetches with the mesh it had."""
    w = synth.refs_water(0, 1000, 31.04, 8, 1, 32)
    good = (w.topo.slt_ljtype, w.topo.slt_charge32)
    want, ctx = _refs_ctx(w, [good]), _refs_ctx(w, [good])
    uvmax, uvsoft, uvcrd = w.uvmax_uvsoft_uvcrd()
    crd = np.concatenate([uvcrd, uvcrd[-1] + np.arange(1.0, 4000.0), [uvcrd[-1]]])
    with pytest.raises(capi.ErError) as ei:
        ctx.set_mesh(np.array([crd.size], np.int32), uvsoft, crd)
    assert ei.value.status == capi.ER_E_ARG
    ctx.clear()
    (ua, ga), = _run(ctx, w, 1)
    (ub, gb), = _run(want, w, 1)
    np.testing.assert_array_equal(ua[0], ub[0])
    for key in ("edens", "ecorr"):
        np.testing.assert_array_equal(ga[key], gb[key])
    ctx.close()
    want.close()


def test_mesh_waits_for_the_run():
    """er_set_mesh after a run and a clear, neither of which waits: the run
    bins with the mesh it began with, so the new one, which starts above every
    energy, halts nothing."""
    w = synth.refs_water(0, 1000, 31.04, 2000, 1, 32)
    ctx = _refs_ctx(w, [(w.topo.slt_ljtype, w.topo.slt_charge32)])
    ctx.set_frame(w.frame(0), w.cell)
    ctx.set_insertions(w.insertions(0))
    ctx.run(capi.ER_BATCHED)
    ctx.sync()
    uvmax, uvsoft, uvcrd = w.uvmax_uvsoft_uvcrd()
    ctx.run(capi.ER_BATCHED)
    ctx.clear()
    ctx.set_mesh(uvmax, uvsoft, 1.0e30 + 1.0e28 * np.arange(uvcrd.size))
    ctx.sync()
    ctx.close()


def test_insertions_device_memory_ends_before_them():
    """er_set_insertions_device on an allocation of fewer insertions than it
    names: er_run refuses, as the copy that it once made did, and goes on with
    the right number; a pointer to page-locked host memory is copied."""
    w = synth.refs_water(0, 1000, 31.04, 40, 1, 32)
    good = (w.topo.slt_ljtype, w.topo.slt_charge32)
    ctx = _refs_ctx(w, [good])
    x = np.ascontiguousarray(w.insertions(0), np.float32)
    ctx.set_frame(w.frame(0), w.cell)
    ctx.set_insertions(x)
    ctx.run(capi.ER_BATCHED)
    want = ctx.uvengy()[0]
    hip = capi.load()  # finds the HIP runtime that it links
    dev = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(dev), ctypes.c_size_t(x[:10].nbytes)) == 0
    try:
        assert hip.hipMemcpy(dev, ctypes.c_void_p(x.ctypes.data), ctypes.c_size_t(x[:10].nbytes), 1) == 0
        for mode in (capi.ER_BATCHED, capi.ER_PLAIN):
            ctx.set_insertions_device(11, dev.value)
            with pytest.raises(capi.ErError) as ei:
                ctx.run(mode)
            assert ei.value.status == capi.ER_E_HIP
        ctx.set_insertions_device(10, dev.value)
        ctx.run(capi.ER_BATCHED)
        np.testing.assert_array_equal(ctx.uvengy()[0], want[:10])
    finally:
        hip.hipFree(dev)
    pinned = torch.from_numpy(x).pin_memory()
    ctx.set_insertions_device(40, pinned.data_ptr())
    ctx.run(capi.ER_BATCHED)
    np.testing.assert_array_equal(ctx.uvengy()[0], want)
    ctx.close()
