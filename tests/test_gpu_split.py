"""Primitive splits of the J/K work items over bra and ket primitive pairs:
from one lane per quartet to the most lanes a quartet may take, with uneven
primitive counts (8-, 6-, 3- and 1-primitive shells), on the class kernels of
segmented and general-contraction pairs and the global-atomic fallback."""
import numpy as np
import pytest

from tests import systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("target_prim", [1, 3, 4096])
@pytest.mark.parametrize("basis,options", [("6-31g*", {}), ("cc-pvdz", {}), ("cc-pvdz", dict(general_contraction=1)),
                                           ("cc-pvdz", dict(deterministic=1)), ("6-31g*", dict(lds_limit=4096))])
def test_primitive_split_matches_oracle(oracle_mod, basis, options, target_prim):
    import torch
    from gradscf_amd import autotune as at
    from gradscf_amd.jk import DirectJKPlan
    _, _, atm, bas, env = systems.tables(systems.water(), basis, cart=True)
    before = at.get_options()
    try:
        at.set_options(**options)
        at.set_schedule(at.Schedule(target_prim=target_prim))
        plan = DirectJKPlan(atm, bas, env, cart=True, cutoff=0.0)
    finally:
        at.set_options(**before)
        at.reset()
    d = systems.random_density(plan.nao, nb=2, seed=31, symmetric=False)
    dd = torch.as_tensor(d, device="cuda")
    ref = oracle_mod.direct_jk(atm, bas, env, d, cart=True, workers=4)
    # the bound of the other J/K tests against the oracle (1e-10 per element)
    assert np.max(np.abs(plan.jk(dd).cpu().numpy() - ref)) < 1e-10
    plan.incore(True)
    assert np.max(np.abs(plan.jk(dd).cpu().numpy() - ref)) < 1e-10
