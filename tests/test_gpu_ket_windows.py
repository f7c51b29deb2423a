"""Ket-side Coulomb sums in LDS windows: chunks of several bras whose kets fit
the window, chunks of more kets than it holds, and chunks of one bra (no
window) give the same bits under integer accumulation, where every quartet adds
the same rounded terms whatever its chunk, and the oracle's values.  The four
densities of one launch take more than half a CU's LDS (512-thread workgroups)
except under lds_limit, where each has a launch of its own."""
import numpy as np
import pytest

from gradscf_amd import molecule as M
from tests import systems

pytestmark = pytest.mark.gpu


def _build(tables, schedule, options, d):
    import torch
    from gradscf_amd import autotune as at
    from gradscf_amd.jk import DirectJKPlan
    before = at.get_options()
    try:
        at.set_options(**options)
        at.set_schedule(at.Schedule(**schedule))
        plan = DirectJKPlan(*tables, cart=True, cutoff=0.0)
        return plan.jk(torch.as_tensor(d, device="cuda")).cpu().numpy()
    finally:
        at.set_options(**before)
        at.reset()


@pytest.mark.parametrize("waters", [1, 8])
def test_windows_add_the_same_terms(oracle_mod, waters):
    # 8 waters: 896 ps pairs, against 682 a window of one density holds
    _, _, *tables = systems.tables(M.water_cluster(waters, seed=3, box=8.0), "6-31g", cart=True)
    d = systems.random_density(oracle_mod.nao(tables[1], True), nb=2, seed=5, symmetric=False)
    outs = [_build(tables, sched, dict(deterministic=1, **opt), d)
            for sched, opt in ((dict(bras_max=1), {}), ({}, {}), (dict(bras_max=2), {}),
                               (dict(chunk_items=65536), {}), (dict(ket_lds=1), {}),
                               (dict(bras_max=256, lds_pack=65536, chunk_items=65536), {}),
                               ({}, dict(lds_limit=16384)))]
    for o in outs[1:]:
        assert np.array_equal(o, outs[0])
    if waters == 1:
        # the bound of the other J/K tests against the oracle (1e-10 per element)
        ref = oracle_mod.direct_jk(*tables, d, cart=True, workers=4)
        assert np.max(np.abs(outs[0] - ref)) < 1e-10
