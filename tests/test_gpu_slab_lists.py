"""Exchange-row slabs folded by one wavefront per row (many rows, short lists)
and by four (few rows, long lists), against builds without slabs."""
import pytest

from gradscf_amd import molecule as M
from tests import systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,waters,basis", [(400, 1, "sto-3g"), (1, 1, "sto-3g"), (1, 6, "cc-pvdz"),
                                                (40, 2, "cc-pvdz")])
@pytest.mark.parametrize("streams", [1, 4])
def test_slab_reduction_matches_atomics(count, waters, basis, streams):
    import torch
    from gradscf_amd import autotune as at
    from gradscf_amd.jk import DirectJKPlan
    specs = [M.water_cluster(waters, seed=i, box=4.0 + 2 * waters) for i in range(min(count, 8))]
    tables = [systems.tables(s, basis, cart=False)[2:] for s in specs]
    tables = [tables[i % len(tables)] for i in range(count)]
    before, out = at.get_options(), []
    try:
        for partial in (1, 0):
            at.set_options(partial_sums=partial, streams=streams, balance=0)
            plan = DirectJKPlan.batch(tables, cart=False, cutoff=1e-10)
            g = torch.Generator(device="cuda").manual_seed(1)
            d = torch.randn((2, plan.nn_total), dtype=torch.float64, device="cuda", generator=g)
            if count == 1:
                d = d.reshape(2, plan.nao, plan.nao)
            out.append([plan.jk(d, symmetric=False)])
            plan.incore(True)
            out[-1].append(plan.jk(d, symmetric=False))
    finally:
        at.set_options(**before)
    for a, b in zip(*out):
        # the same terms summed in another order
        assert float((a - b).abs().max()) < 1e-12 * max(1.0, float(b.abs().max()))
