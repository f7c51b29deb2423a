"""Plans and packed integrals whose lists pass the 2^32 work items of one
launch."""
import numpy as np
import pytest

from gradscf_amd.molecule import parse_molecule_spec
from tests import systems

pytestmark = pytest.mark.gpu


def hydrogens(n):
    """STO-3G tables of n H atoms 1.5 Angstrom apart on a shaken grid."""
    rng = np.random.default_rng(1)
    grid = [(i, j, k) for i in range(8) for j in range(8) for k in range(8)][:n]
    atoms = [("H", tuple(1.5 * np.array(x) + rng.uniform(-0.2, 0.2, 3))) for x in grid]
    _, _, *tables = systems.tables(parse_molecule_spec(atoms), "sto-3g", cart=True)
    return tables


def test_unscreened_plan_past_one_launch():
    import torch
    from gradscf_amd.jk import DirectJKPlan
    n, cutoff = 433, 1e-13
    tables = hydrogens(n)
    d = torch.as_tensor(systems.random_density(n, seed=3), device="cuda")
    screened = DirectJKPlan(*tables, cart=True, cutoff=cutoff).jk(d).cpu()
    plan = DirectJKPlan(*tables, cart=True, cutoff=0.0)
    assert plan.info["nquartets"] > 2 ** 32
    out = plan.jk(d).cpu()
    # every quartet the screened plan leaves out is below the cutoff, and an
    # element sums at most n^2 of them times a density element
    assert float((out - screened).abs().max()) < n * n * cutoff * float(d.abs().max())


def test_packed_integrals_past_one_launch():
    import torch
    from gradscf_amd.jk import DirectJKPlan, packed_eri, packed_jk
    n = 220
    tables = hydrogens(n)
    eri = packed_eri(*tables, cart=True)
    d = torch.as_tensor(systems.random_density(n, seed=4), device="cuda")
    ref = DirectJKPlan(*tables, cart=True, cutoff=0.0).jk(d)
    # the bound of the other J/K comparisons (1e-10 per element)
    assert float((torch.stack(packed_jk(eri, d)) - ref).abs().max()) < 1e-10


def test_auxiliary_integrals_past_one_launch():
    """500 orbital s shells of six primitives against 2200 auxiliary ones: the
    rows of the first and the last auxiliary shells are those of a call with
    these alone."""
    import torch
    from gradscf_amd.density_fitting import evaluate
    rng = np.random.default_rng(2)
    norb, naux, part = 500, 2200, 40
    atm = np.zeros((8, 6), np.int32)
    atm[:, 0] = 1
    atm[:, 1] = 20 + 3 * np.arange(8)
    atm[:, 2] = 1
    orb_exp = 0.3 * 2.5 ** np.arange(6)
    aux_exp = rng.uniform(0.2, 4.0, naux)
    env = np.concatenate([np.zeros(20), rng.uniform(-0.5, 0.5, 24), orb_exp, rng.uniform(0.2, 1.0, 6), aux_exp,
                          np.ones(naux)])

    def bas(aux):
        rows = [[i % 8, 0, 6, 1, 0, 44, 50, 0] for i in range(norb)]
        return np.array(rows + [[i % 8, 0, 1, 1, 0, 56 + i, 56 + naux + i, 0] for i in aux], np.int32)

    def three(aux):
        return evaluate(atm, bas(aux), env, (len(aux), norb * (norb + 1) // 2), layout=3, cart=True, split=norb)

    whole = three(range(naux))
    assert torch.equal(whole[:part], three(range(part)))
    assert torch.equal(whole[-part:], three(range(naux - part, naux)))


def test_one_electron_matrices_past_one_launch():
    """11700 distant s functions: 6.8e7 pairs, one wavefront each."""
    import torch
    from gradscf_amd.jk import DirectJKPlan
    n, a = 11700, 0.4
    grid = np.stack(np.unravel_index(np.arange(n), (23, 23, 23)), -1) * 60.0
    atm = np.zeros((n, 6), np.int32)
    atm[0, 0] = 1
    atm[:, 1] = 20 + 3 * np.arange(n)
    atm[:, 2] = 1
    env = np.concatenate([np.zeros(20), grid.ravel(), [a, (2 * a / np.pi) ** 0.75 * (4 * np.pi) ** 0.5]])
    bas = np.zeros((n, 8), np.int32)
    bas[:, 0] = np.arange(n)
    bas[:, 2:4] = 1
    bas[:, 5:7] = len(env) - 2, len(env) - 1
    plan = DirectJKPlan(atm, bas, env, cart=True, cutoff=1e3)
    s, t, v = plan.int1e()
    dist = torch.as_tensor(np.sqrt((grid ** 2).sum(-1)), device="cuda")
    nuc = -torch.erf((2 * a) ** 0.5 * dist) / dist
    nuc[0] = -2 * (2 * a / np.pi) ** 0.5
    # a few rounding errors of the (diagonal) value; all else is exactly zero
    for m, ref in ((s, torch.ones_like(nuc)), (t, torch.full_like(nuc, 1.5 * a)), (v, nuc)):
        assert float((m.diagonal() - ref).abs().max()) < 1e-13
        assert int(torch.count_nonzero(m)) == n


def _p_shells(n, exponent, coords):
    """Tables of n single-primitive p shells with one exponent."""
    atm = np.zeros((len(coords), 6), np.int32)
    atm[:, 0] = 1
    atm[:, 1] = 20 + 3 * np.arange(len(coords))
    atm[:, 2] = 1
    env = np.concatenate([np.zeros(20), coords.ravel(), [exponent, 1.0]])
    bas = np.zeros((n, 8), np.int32)
    bas[:, 0] = np.arange(n) % len(coords)
    bas[:, 1:4] = 1
    bas[:, 5:7] = len(env) - 2, len(env) - 1
    return atm, bas, env


def test_derivatives_past_one_launch():
    """(pp|pp) derivatives of 260 p shells: 5.8e8 quartets of nine ket
    components each, against central differences of J and K."""
    import torch
    from gradscf_amd.jk import DirectJKPlan
    n, alpha, h = 260, 0.8, 1e-4
    rng = np.random.default_rng(5)
    grid = np.stack(np.unravel_index(np.arange(260), (7, 7, 7)), -1) * 1.2 + rng.uniform(-0.2, 0.2, (260, 3))
    d, cj, ck = (torch.as_tensor(x, device="cuda") for x in systems.random_density(3 * n, nb=3, seed=12))
    plan = DirectJKPlan(*_p_shells(n, alpha, grid), cart=True, cutoff=0.0)
    assert plan.info["nquartets"] * 9 > 2 ** 32

    def energy(exponent, coords):
        j, k = DirectJKPlan(*_p_shells(n, exponent, coords), cart=True, cutoff=0.0).jk(d)
        return float((cj * j).sum() + (ck * k).sum())

    u = rng.normal(size=grid.shape)
    grad = plan.jk_geometry_vjp(d, cj, ck).cpu().numpy()
    slope = (energy(alpha, grid + h * u) - energy(alpha, grid - h * u)) / (2 * h)
    # central differences: a third derivative times h^2 / 6
    assert abs((grad * u).sum() - slope) < 1e-5 * np.abs(grad * u).sum()
    env_grad = plan.jk_param_vjp(d, cj, ck)
    slope = (energy(alpha + h, grid) - energy(alpha - h, grid)) / (2 * h)
    assert abs(float(env_grad[-2]) - slope) < 1e-5 * abs(slope)
