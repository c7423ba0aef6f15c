"""Calls between runs: what er_get_flceng gives after the solute list grows."""
import numpy as np
import pytest

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
