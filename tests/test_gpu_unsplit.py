"""Primitive quartets of one lane: a system with enough quartets in every class
for one lane per contracted quartet (a small one is split until it fills the
device, whatever target_prim allows), against the most lanes a quartet may
take.  (The plans differ: their chunk lists, and so their device bytes, do.)"""
import pytest

from gradscf_amd import molecule as M
from tests import systems

pytestmark = pytest.mark.gpu

FILL_LANES = 32768  # lanes a class is filled to before target_prim counts


def _prims(bas, l):
    """Primitives of all segmented shells of angular momentum l."""
    rows = bas[bas[:, 1] == l]
    return int((rows[:, 2] * rows[:, 3]).sum()), int(rows[:, 2].max())


@pytest.mark.parametrize("basis,options", [("6-31g*", {}), ("cc-pvdz", {}), ("cc-pvdz", dict(general_contraction=1)),
                                           ("cc-pvdz", dict(deterministic=1)), ("6-31g*", dict(lds_limit=4096))])
def test_one_lane_per_quartet(basis, options):
    import torch
    from gradscf_amd import autotune as at
    from gradscf_amd.jk import DirectJKPlan
    _, _, *tables = systems.tables(M.water_cluster(12, seed=12, box=5.5), basis, cart=True)
    # every class of s shells passes the fill at one lane per quartet
    total, largest = _prims(tables[1], 0)
    assert (total * total / 2) ** 2 / 2 > FILL_LANES * largest ** 4
    before, out, held = at.get_options(), [], []
    try:
        at.set_options(**dict(options, balance=0))
        for target in (4096, 1):
            at.set_schedule(at.Schedule(target_prim=target))
            plan = DirectJKPlan(*tables, cart=True, cutoff=0.0)
            held.append(plan.device_bytes())
            d = torch.as_tensor(systems.random_density(plan.nao, nb=2, seed=31, symmetric=False), device="cuda")
            out.append(plan.jk(d))
            plan.incore(True)
            out.append(plan.jk(d))
            del plan
    finally:
        at.set_options(**before)
        at.reset()
    assert held[0] != held[1]
    # the bound of the other J/K comparisons (1e-10 per element), each side
    for o in out[1:]:
        assert float((o - out[0]).abs().max()) < 2e-10
