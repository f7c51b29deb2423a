"""One-electron matrices and their gradient where the wavefront-per-pair kernels
change shape: one nucleus lane, nuclei counts at and around the 64 lanes of a
wavefront, and more shell pairs than the persistent gradient grid has
wavefronts."""
import numpy as np
import pytest

from tests import systems

pytestmark = pytest.mark.gpu

# one-primitive shells keep the oracle's quadrature affordable at 65 nuclei
BASIS = {"H": [[0, [0.7, 1.0]]], "O": [[0, [5.0, 0.4], [1.1, 0.7]], [1, [0.9, 1.0]], [2, [1.2, 1.0]]]}


def _chain(nuclei):
    rng = np.random.default_rng(nuclei)
    atoms = [("O", (0.0, 0.0, 0.0))] + [("H", (1.0 + 0.9 * i, *rng.normal(scale=0.3, size=2)))
                                        for i in range(nuclei - 1)]
    from gradscf_amd.molecule import parse_molecule_spec
    return parse_molecule_spec(atoms)


@pytest.mark.parametrize("cart", [True, False])
@pytest.mark.parametrize("nuclei", [1, 3, 64, 65])
def test_core_matrices_match_oracle(oracle_mod, nuclei, cart):
    from gradscf_amd.jk import DirectJKPlan
    _, _, atm, bas, env = systems.tables(_chain(nuclei), BASIS, cart=cart)
    plan = DirectJKPlan(atm, bas, env, cart=cart, cutoff=1e-12)
    for got, ref in zip(plan.int1e(), oracle_mod.int1e(atm, bas, env, cart)):
        # FP64 rounding over at most 65 nuclei of charge <= 8
        assert np.max(np.abs(got.cpu().numpy() - ref)) < 1e-12 * max(1.0, np.max(np.abs(ref)))


@pytest.mark.parametrize("nuclei", [3, 65, 90])
def test_core_gradient_matches_differences(nuclei):
    """Five-point differences (h = 1e-3 bohr) of sum D (T + V) - W S along a nuclear
    row and a basis-centre row; |E| < 1e4, so rounding leaves about 1e-9."""
    import torch
    from gradscf_amd.jk import DirectJKPlan
    _, _, atm, bas, env = systems.tables(_chain(nuclei), BASIS, cart=False)
    plan = DirectJKPlan(atm, bas, env, cart=False, cutoff=1e-12)
    d, w = (torch.as_tensor(systems.random_density(plan.nao, seed=s)[0], device="cuda") for s in (5, 6))
    rows = plan.int1e_gradient(d, w).cpu().numpy()

    def energy(slot, h):
        e = env.copy()
        e[slot] += h
        s, t, v = DirectJKPlan(atm, bas, e, cart=False, cutoff=1e-12).int1e()
        return float((d * (t + v) - w * s).sum())

    h = 1e-3
    for row, x in ((0, 1), (nuclei, 2), (nuclei - 1, 0)):
        f = [energy(int(atm[row, 1]) + x, k * h) for k in (-2, -1, 1, 2)]
        assert abs((f[0] - 8 * f[1] + 8 * f[2] - f[3]) / (12 * h) - rows[row, x]) < 1e-7
