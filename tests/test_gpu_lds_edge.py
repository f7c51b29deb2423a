"""Slots that fit the LDS limit without the bra's 80-byte record and exceed it
with the record: such a class keeps the LDS route (and its integrals can be
kept in core), reading its primitives from memory instead of staging them."""
import numpy as np
import pytest

from tests import systems

pytestmark = pytest.mark.gpu

ROW, RECORD, STAGED = 8, 80, 48  # bytes: a column of one row, a bra's record, a staged primitive pair


def _tables(nprim, extra):
    """Two s shells of nprim primitives and `extra` of one on two centres."""
    rng = np.random.default_rng(nprim)
    atm = np.zeros((2, 6), np.int32)
    atm[:, 0] = 1
    atm[:, 1] = 20, 23
    atm[:, 2] = 1
    counts = [nprim, nprim] + [1] * extra
    env, bas = [0.0] * 20 + list(rng.uniform(-0.5, 0.5, 6)), []
    for i, k in enumerate(counts):
        bas.append([i % 2, 0, k, 1, 0, len(env), len(env) + k, 0])
        env += list(0.3 * 1.8 ** np.arange(k)) + list(rng.uniform(0.2, 1.0, k))
    return atm, np.array(bas, np.int32), np.array(env)


@pytest.mark.parametrize("deterministic", [0, 1])
@pytest.mark.parametrize("nprim", [8, 9])
def test_record_does_not_cost_the_lds_route(oracle_mod, nprim, deterministic):
    import torch
    from gradscf_amd import autotune as at
    from gradscf_amd.jk import DirectJKPlan
    limit = 4096
    # a slot: two rows of n columns, nine block values, staged pairs, record
    fixed = 9 * 8 + nprim * nprim * STAGED + RECORD
    n = (limit - fixed) // (2 * ROW) + 1
    slot = 2 * ROW * n + fixed
    assert limit < slot <= limit + RECORD - 8
    tables = _tables(nprim, n - 2)
    before = at.get_options()
    try:
        at.set_options(lds_limit=limit, deterministic=deterministic, balance=0)
        plan = DirectJKPlan(*tables, cart=True, cutoff=0.0)
    finally:
        at.set_options(**before)
    assert plan.nao == n and plan.info["classes_global_atomic"] == 0
    d = systems.random_density(n, nb=1, seed=3, symmetric=False)
    ref = oracle_mod.direct_jk(*tables, d, cart=True, workers=4)
    out = plan.jk(torch.as_tensor(d, device="cuda")).cpu().numpy()
    # the bound of the other J/K tests against the oracle, for integrals of this size
    assert np.max(np.abs(out - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
    plan.incore(True)
    kept = plan.jk(torch.as_tensor(d, device="cuda")).cpu().numpy()
    assert np.max(np.abs(kept - ref)) < 1e-10 * max(1.0, np.max(np.abs(ref)))
    if deterministic:
        assert np.array_equal(kept, out)
