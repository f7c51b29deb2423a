"""Density-fitting integrals of every (orbital class, auxiliary l) combination
against the oracle's four-centre ERIs with the unit function in the last slot:
contracted and general-contraction orbital shells, auxiliary shells s..g with
one to five primitives, molecules whose task counts leave partly filled blocks.
The oracle transforms shells up to d, so spherical f and g shells are left to
the comparison with libcint's integrals."""
import numpy as np
import pytest

from gradscf_amd import molecule as M
from tests import systems
from tests.test_gpu_df import _tables
from tests.test_oracle import _with_unit

pytestmark = pytest.mark.gpu


def _blocks(ao, shells):
    return np.ix_(*[np.arange(ao[s], ao[s + 1]) for s in shells])


@pytest.mark.parametrize("cart", [True, False])
@pytest.mark.parametrize("aux,orbital,waters", [("def2-universal-jkfit", "cc-pvdz", 1),
                                                ("cc-pvdz-jkfit", "6-31g*", 2), ("cc-pvdz-jkfit", "sto-3g", 1)])
def test_auxiliary_integrals_match_unit_function_eris(oracle_mod, aux, orbital, waters, cart):
    from gradscf_amd.density_fitting import evaluate
    from gradscf_amd.packing import ao_offsets
    spec = M.water_monomer() if waters == 1 else systems.water_dimer()
    plan, _, _, atm, bas, env = _tables(aux, cart, spec=spec, orbital=orbital)
    n, m, split = plan.orbital.nao(), plan.auxiliary.nao(), plan.split
    ao = ao_offsets(bas, cart)
    two = evaluate(atm, bas, env, (m, m), layout=2, cart=cart, split=split).cpu().numpy()
    packed = evaluate(atm, bas, env, (m, n * (n + 1) // 2), layout=3, cart=cart, split=split).cpu().numpy()
    assert np.array_equal(two, two.T)
    three = np.zeros((n, n, m))
    i, j = np.tril_indices(n)
    three[i, j] = three[j, i] = packed.T
    rng = np.random.default_rng(17)
    ls = bas[:, 1]

    def pick(shells, l):
        return int(rng.choice(shells[ls[shells] == l]))

    orb, fit = np.arange(split), np.arange(split, len(bas))
    fit = fit[ls[fit] <= (4 if cart else 2)]
    for lk in np.unique(ls[fit]):
        k = pick(fit, lk)
        a2, b2, e2 = _with_unit(atm, bas, env, int(bas[k, 0]))
        u = len(b2) - 1
        for la in np.unique(ls[orb]):
            for lb in np.unique(ls[orb]):
                s, t = pick(orb, la), pick(orb, lb)
                ref = oracle_mod.eri_block((s, t, k, u), a2, b2, e2, cart)[..., 0]
                got = three[_blocks(ao, (s, t))][:, :, ao[k] - n:ao[k + 1] - n]
                # FP64 rounding of a sum over at most 64 primitive pairs
                assert np.max(np.abs(got - ref)) < 1e-12 * max(1.0, np.max(np.abs(ref))), (s, t, k)
        for lq in np.unique(ls[fit]):
            q = pick(fit, lq)
            a3, b3, e3 = _with_unit(a2, b2, e2, int(bas[q, 0]))
            ref = oracle_mod.eri_block((k, u, q, len(b3) - 1), a3, b3, e3, cart)[:, 0, :, 0]
            got = two[ao[k] - n:ao[k + 1] - n, ao[q] - n:ao[q + 1] - n]
            assert np.max(np.abs(got - ref)) < 1e-12 * max(1.0, np.max(np.abs(ref))), (k, q)
