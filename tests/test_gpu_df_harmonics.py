"""Spherical density-fitting integrals up to g against the Cartesian ones (whose
blocks are compared with the oracle elsewhere), transformed by real solid
harmonics fitted here from associated Legendre functions."""
import math

import numpy as np
import pytest
from scipy.special import lpmv

from gradscf_amd import molecule as M
from tests.test_gpu_df import _tables


def _components(l):
    """Cartesian exponents in libcint's order."""
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _harmonics(l):
    """(2l + 1, components): r^l Y_lm, m = -l .. l, as polynomials in x, y, z
    (no Condon-Shortley phase; l < 2: the components themselves)."""
    if l < 2:
        return np.eye(2 * l + 1)
    rng = np.random.default_rng(l)
    p = rng.normal(size=(200, 3))
    r = np.linalg.norm(p, axis=1)
    phi = np.arctan2(p[:, 1], p[:, 0])
    monomials = np.stack([p[:, 0] ** x * p[:, 1] ** y * p[:, 2] ** z for x, y, z in _components(l)], 1)
    rows = []
    for m in range(-l, l + 1):
        a = abs(m)
        norm = math.sqrt((2 * l + 1) / (4 * math.pi) * math.factorial(l - a) / math.factorial(l + a))
        v = (-1) ** a * norm * lpmv(a, l, p[:, 2] / r) * r ** l
        if m:
            v = v * math.sqrt(2) * (np.sin(a * phi) if m < 0 else np.cos(a * phi))
        rows.append(np.linalg.lstsq(monomials, v, rcond=None)[0])
    return np.stack(rows)


def _transform(bas):
    blocks = [_harmonics(int(l)) for row in bas for l in [row[1]] * int(row[3])]
    out = np.zeros((sum(b.shape[0] for b in blocks), sum(b.shape[1] for b in blocks)))
    i = j = 0
    for b in blocks:
        out[i:i + b.shape[0], j:j + b.shape[1]] = b
        i, j = i + b.shape[0], j + b.shape[1]
    return out


@pytest.mark.parametrize("l", [2, 3, 4])
def test_harmonics_are_orthonormal_and_harmonic(l):
    t, comps = _harmonics(l), _components(l)

    def moment(e):
        """Mean over the sphere of x^i y^j z^k."""
        if any(k % 2 for k in e):
            return 0.0
        f = lambda k: math.prod(range(k - 1, 0, -2))  # noqa: E731
        return f(e[0]) * f(e[1]) * f(e[2]) / math.prod(range(sum(e) + 1, 0, -2))

    gram = np.array([[moment([p + q for p, q in zip(a, b)]) for b in comps] for a in comps])
    assert np.allclose(4 * math.pi * t @ gram @ t.T, np.eye(2 * l + 1), atol=1e-12)
    assert t.shape == (2 * l + 1, len(comps))


@pytest.mark.gpu
@pytest.mark.parametrize("aux,orbital", [("def2-universal-jkfit", "cc-pvdz"), ("cc-pvdz-jkfit", "6-31g*")])
def test_spherical_auxiliary_integrals_are_transformed_cartesian_ones(aux, orbital):
    from gradscf_amd.density_fitting import evaluate

    def integrals(cart):
        plan, _, _, atm, bas, env = _tables(aux, cart, spec=M.water_monomer(), orbital=orbital)
        n, m, split = plan.orbital.nao(), plan.auxiliary.nao(), plan.split
        kw = dict(cart=cart, split=split)
        two = evaluate(atm, bas, env, (m, m), layout=2, **kw).cpu().numpy()
        packed = evaluate(atm, bas, env, (m, n * (n + 1) // 2), layout=3, **kw).cpu().numpy()
        three = np.zeros((m, n, n))
        i, j = np.tril_indices(n)
        three[:, i, j] = three[:, j, i] = packed
        return two, three, bas, split

    two, three, bas, split = integrals(True)
    if aux == "def2-universal-jkfit":
        assert {3, 4} <= set(bas[split:, 1])
    to, ta = _transform(bas[:split]), _transform(bas[split:])
    two_s, three_s, _, _ = integrals(False)
    ref2 = ta @ two @ ta.T
    ref3 = np.einsum("pP,Pab,qa,rb->pqr", ta, three, to, to, optimize=True)
    # rounding of sums of at most 6 x 6 x 6 terms
    assert np.max(np.abs(two_s - ref2)) < 1e-12 * max(1.0, np.max(np.abs(ref2)))
    assert np.max(np.abs(three_s - ref3)) < 1e-12 * max(1.0, np.max(np.abs(ref3)))
