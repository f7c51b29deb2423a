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
