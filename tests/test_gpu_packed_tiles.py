"""Packed ERIs over every class and primitive split against the oracle, and packed
J/K at the edges of its tiles: one AO, row groups of eight that do and do not
divide the AO count, the 64 lanes of a wavefront, and AO counts past the row
group that fits in LDS.  The J/K inputs are outer products v(ab, cd) = x_ab x_cd,
whose J and K are X (X . D) and X D X."""
import numpy as np
import pytest

from tests import systems
from tests.test_gpu_packed import _s8_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,cart", [("cc-pvdz", False), ("cc-pvdz", True), ("sto-3g", True)])
def test_packed_eri_classes_match_oracle(oracle_mod, basis, cart):
    from gradscf_amd.jk import packed_eri
    _, _, atm, bas, env = systems.tables(systems.water(), basis, cart=cart)
    full = oracle_mod.full_eri(atm, bas, env, cart=cart)
    n = full.shape[0]
    s8 = packed_eri(atm, bas, env, cart=cart).cpu().numpy()
    # the bound of the other packed-ERI comparison
    assert np.max(np.abs(s8[_s8_indices(n)] - full)) < 1e-12
    s4 = packed_eri(atm, bas, env, cart=cart, aosym="s4").cpu().numpy()
    rows, cols = np.tril_indices(len(s4))
    assert np.array_equal(s4, s4.T) and np.array_equal(s4[rows, cols], s8)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65, 130, 456])
def test_packed_jk_tiles(n):
    import torch
    from gradscf_amd.jk import packed_jk
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n * (n + 1) // 2, dtype=torch.float64, device="cuda", generator=g)
    eri = torch.empty(len(x) * (len(x) + 1) // 2, dtype=torch.float64, device="cuda")
    for r in range(len(x)):
        eri[r * (r + 1) // 2:(r + 1) * (r + 2) // 2] = x[r] * x[:r + 1]
    i, j = (torch.as_tensor(t, device="cuda") for t in np.tril_indices(n))
    full = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    full[i, j] = full[j, i] = x
    nb = 1 if n > 200 else 2
    d = torch.randn((nb, n, n), dtype=torch.float64, device="cuda", generator=g)
    gj, gk = packed_jk(eri, d)
    for b in range(nb):
        # rounding: a few hundred ulp of the sum of absolute terms
        top_j = full.abs() * (full.abs() * d[b].abs()).sum()
        top_k = full.abs() @ d[b].abs() @ full.abs()
        assert bool(((gj[b] - full * (full * d[b]).sum()).abs() <= 1e-13 * top_j).all())
        assert bool(((gk[b] - full @ d[b] @ full).abs() <= 1e-13 * top_k).all())
        assert torch.equal(gj[b], gj[b].T)
