"""The `balance` option: with balance=1 set, plan creation measures the classes
of short builds too (its probe builds leave the plan a workspace, which the
plan's device bytes show); with balance=0 it makes no build."""
import pytest

from tests import systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [False, True])
def test_balance_that_was_set_measures_short_builds(batch):
    from gradscf_amd import autotune as at
    from gradscf_amd.jk import DirectJKPlan
    _, _, *tables = systems.tables(systems.water_dimer(), "cc-pvdz", cart=False)
    before, held = at.get_options(), {}
    try:
        for balance in (0, 1):
            at.set_options(balance=balance)
            plan = (DirectJKPlan.batch([tables, tables], cart=False) if batch
                    else DirectJKPlan(*tables, cart=False))
            held[balance] = plan.device_bytes()
    finally:
        at.set_options(**before)
    assert held[1] > held[0]
