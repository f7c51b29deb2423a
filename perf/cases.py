"""The work a user of the engine has it do, as measurable cases.

Every case is one pass through the public entry points with what a program has
in hand before the call (tables, a plan, densities) made from a seed:

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  the program's state before the call
  run(state)           one pass, returning its whole outputs
  work(case)           bytes and operations one pass cannot do without
  exact(case, seed)    what run returns, by plain 64-bit torch: McMurchie-Davidson
                       Hermite integrals over whole shell-pair classes (the engine
                       itself uses Rys quadrature), derivatives by autograd

Kinds of pass: "jk" (J/K of one plan, the SCF iteration's call), "direct" (the
reference-style direct_jk call on tables, host checks included), "incore" (J/K from
stored integrals), "batch" (J/K of many molecules in one plan), "geometry" and
"basis" (the coordinate and the exponent/coefficient derivative of the J/K energy),
"auxiliary" (density-fitting integrals), "packed" (packed ERIs of a small molecule
and J/K from them), "core" (one-electron matrices and their gradient) and "fresh" (a
new geometry: plan, core matrices and J/K, the first step of every new SCF).
"""
import math

import numpy as np
import torch

from gradscf_amd import molecule as M
from gradscf_amd import roofline
from gradscf_amd.basis import prepare_basis
from gradscf_amd.density_fitting import make_auxiliary_plan
from gradscf_amd.jk import DirectJKPlan, direct_jk, packed_eri, packed_jk
from gradscf_amd.packing import ao_offsets, pack

BASES = ("sto-3g", "6-31g", "6-31g*", "cc-pvdz")


def _case(kind, system, size, basis, cart, cutoff=0.0, nb=1, symmetric=True, with_j=True, with_k=True, name=None):
    c = dict(kind=kind, system=system, size=size, basis=basis, cart=cart, cutoff=cutoff, nb=nb,
             symmetric=symmetric, with_j=with_j, with_k=with_k)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest J/K call of a small-molecule SCF: latency and launches only
        _case("jk", "water", 1, "6-31g", True, name="jk water 6-31g"),
        # the headline J/K build: one SCF iteration of a 16-molecule cluster
        _case("jk", "water", 16, "cc-pvdz", False, 1e-12, name="jk (H2O)16 cc-pvdz"),
        # an elongated molecule in a Cartesian Pople basis: many screened pairs
        _case("jk", "alkane", 20, "6-31g*", True, 1e-12, name="jk C20H42 6-31g*"),
        # two nonsymmetric densities through the reference's call (response equations)
        _case("direct", "water", 7, "cc-pvdz", False, 1e-12, nb=2, symmetric=False, name="direct (H2O)7 nonsym"),
        # many small molecules at once: a batched SCF iteration
        _case("batch", "water", 64, "6-31g*", True, 1e-12, name="batch 64 clusters"),
        # an SCF iteration that digests integrals kept in HBM
        _case("incore", "water", 8, "cc-pvdz", False, 1e-12, name="incore (H2O)8 cc-pvdz"),
        # nuclear forces: the coordinate derivative (unscreened, as it requires)
        _case("geometry", "water", 5, "cc-pvdz", False, name="geometry (H2O)5 cc-pvdz"),
        # basis optimisation: every exponent and coefficient derivative
        _case("basis", "water", 3, "cc-pvdz", False, name="basis (H2O)3 cc-pvdz"),
        # density fitting: the metric and the three-centre integrals of one geometry
        _case("auxiliary", "water", 4, "cc-pvdz", False, name="auxiliary (H2O)4 jkfit"),
        # the small-molecule route: packed ERIs, then J/K from them
        _case("packed", "water", 2, "6-31g*", True, name="packed (H2O)2 6-31g*"),
        # S, T, V of an SCF set-up and the one-electron part of the forces
        _case("core", "water", 16, "cc-pvdz", False, name="core (H2O)16 cc-pvdz"),
        # a new geometry (dynamics, optimisation): plan, core matrices, first J/K
        _case("fresh", "water", 3, "6-31g*", True, 1e-12, name="fresh (H2O)3 6-31g*"),
    ]


# largest molecule count drawn per kind (carbons: 20)
_LARGEST = {"jk": 16, "direct": 7, "batch": 64, "incore": 8, "geometry": 5, "basis": 3, "auxiliary": 4,
            "packed": 2, "core": 16, "fresh": 3}


def draw(rng):
    kind = rng.choice(sorted(_LARGEST))
    top = _LARGEST[kind]
    size = min(top, int(math.exp(rng.uniform(0.0, math.log(top + 1.0)))))
    system = "water"
    basis = rng.choice(BASES)
    cart = rng.random() < 0.5
    if kind == "auxiliary":
        basis = "cc-pvdz"
    if kind == "batch":
        size = max(2, size)
        basis, cart = rng.choice(BASES[:3]), True
    if kind in ("jk", "direct", "incore", "core") and rng.random() < 0.3:
        system = "alkane"
        size = rng.randint(2, 20 if kind in ("jk", "core") else 8)
        basis, cart = rng.choice(BASES[:3]), True
    cutoff = rng.choice((1e-10, 1e-11, 1e-12)) if kind in ("jk", "direct", "incore", "batch", "fresh") else 0.0
    nb, symmetric = 1, True
    if kind in ("jk", "direct", "incore") and size <= 8:
        nb = rng.choice((1, 1, 2))
        symmetric = rng.random() < 0.6
    with_j = with_k = True
    if kind in ("jk", "direct", "incore", "geometry", "basis"):
        with_j, with_k = rng.choice(((True, True), (True, True), (True, False), (False, True)))
    return _case(kind, system, size, basis, cart, cutoff, nb, symmetric, with_j, with_k)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _specs(case, seed):
    """Molecules at the geometries of `seed`: random clusters at the density of
    liquid water, alkane chains with thermal displacements (0.03 bohr)."""
    if case["system"] == "alkane":
        spec = M.linear_alkane(case["size"])
        move = np.random.default_rng(seed).normal(scale=0.03, size=spec.coords_bohr.shape)
        return [M.MoleculeSpec(spec.symbols, spec.coords_bohr + move)]
    if case["kind"] == "batch":
        sizes = np.random.default_rng(256).integers(1, 9, size=case["size"])
    else:
        sizes = [case["size"]]
    return [M.water_cluster(int(n), seed=1000 * seed + i, box=4.8 * n ** (1.0 / 3.0)) for i, n in enumerate(sizes)]


def _tables(case, seed):
    out = []
    for spec in _specs(case, seed):
        topology, parameters = prepare_basis(spec, case["basis"], cart=case["cart"])
        out.append(pack(topology, parameters))
    return out


def _auxiliary(case, seed):
    (spec,) = _specs(case, seed)
    topology, parameters = prepare_basis(spec, case["basis"], cart=case["cart"])
    aux_topology, aux_parameters = prepare_basis(spec, case["basis"] + "-jkfit", cart=case["cart"])
    return make_auxiliary_plan(topology, aux_topology), parameters, aux_parameters


def _matrix(table, cart, rng, symmetric=True):
    """A density-like matrix over the molecule's AOs: diagonal of order one, off-diagonal
    elements that decay with the distance between their centres."""
    atm, bas, env = table
    ao = ao_offsets(bas, cart)
    centre = np.concatenate([np.repeat(env[atm[row[0], 1]:atm[row[0], 1] + 3][None], ao[i + 1] - ao[i], axis=0)
                             for i, row in enumerate(bas)])
    n = len(centre)
    d = np.linalg.norm(centre[:, None] - centre[None], axis=-1)
    x = (0.3 * rng.normal(size=(n, n)) + 0.6 * np.eye(n)) * np.exp(-0.5 * d)
    return 0.5 * (x + x.T) if symmetric else x


def _matrices(case, seed, tables):
    rng = np.random.default_rng([seed, 7])
    if case["kind"] == "batch":
        return np.concatenate([_matrix(t, case["cart"], rng).reshape(-1) for t in tables])[None]
    return np.stack([_matrix(tables[0], case["cart"], rng, case["symmetric"]) for _ in range(case["nb"])])


def _cotangents(case, d):
    """The J/K part of the RHF energy, 1/2 tr(D J) - 1/4 tr(D K)."""
    return (0.5 * d if case["with_j"] else None), (-0.25 * d if case["with_k"] else None)


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "auxiliary":
        state["plan"], state["parameters"], state["aux"] = _auxiliary(case, seed)
        return state
    tables = _tables(case, seed)
    state["tables"] = tables[0]
    state["density"] = torch.as_tensor(_matrices(case, seed, tables)).cuda()
    if kind == "core":
        rng = np.random.default_rng([seed, 8])
        state["weighted"] = torch.as_tensor(_matrix(tables[0], case["cart"], rng)).cuda()
    if kind in ("geometry", "basis"):
        state["cotangents"] = _cotangents(case, state["density"][0])
    if kind == "batch":
        state["plan"] = DirectJKPlan.batch(tables, cart=case["cart"], cutoff=case["cutoff"])
    elif kind in ("jk", "incore", "geometry", "basis", "core"):
        state["plan"] = DirectJKPlan(*tables[0], cart=case["cart"], cutoff=case["cutoff"])
    if kind == "incore":
        state["plan"].incore(True)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("jk", "incore", "batch"):
        return state["plan"].jk(state["density"], symmetric=case["symmetric"], validate=False,
                                with_j=case["with_j"], with_k=case["with_k"])
    if kind == "direct":
        return direct_jk(*state["tables"], state["density"], cart=case["cart"], cutoff=case["cutoff"],
                         with_j=case["with_j"], with_k=case["with_k"])
    if kind == "geometry":
        return state["plan"].jk_geometry_vjp(state["density"][0], *state["cotangents"])
    if kind == "basis":
        return state["plan"].jk_param_vjp(state["density"][0], *state["cotangents"])
    if kind == "auxiliary":
        return state["plan"].evaluate(state["parameters"], state["aux"])
    if kind == "packed":
        eri = packed_eri(*state["tables"], cart=case["cart"])
        return eri, packed_jk(eri, state["density"])
    if kind == "core":
        s, t, v = state["plan"].int1e()
        return s, t, v, state["plan"].int1e_gradient(state["density"][0], state["weighted"])
    plan = DirectJKPlan(*state["tables"], cart=case["cart"], cutoff=case["cutoff"])
    return plan.int1e(), plan.jk(state["density"], symmetric=True, validate=False)


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _schwarz(table):
    """Shell-pair bounds sqrt((ss|ss)) of the shells' radial parts: close enough to
    count the quartets that survive the cutoff."""
    atm, bas, env = table
    rows = [(env[r[5]:r[5] + r[2]], np.abs(env[r[6]:r[6] + r[2] * r[3]].reshape(r[3], r[2])).max(axis=0),
             env[atm[r[0], 1]:atm[r[0], 1] + 3]) for r in bas]
    q = np.zeros((len(rows), len(rows)))
    for i, (a, ca, ra) in enumerate(rows):
        for j, (b, cb, rb) in enumerate(rows[:i + 1]):
            p = a[:, None] + b[None]
            k = ca[:, None] * cb[None] * 0.08 * np.exp(-a[:, None] * b[None] / p * float(np.sum((ra - rb) ** 2)))
            q[i, j] = q[j, i] = np.sum(k * np.sqrt(2 * math.pi ** 2.5 / (p * p * np.sqrt(2 * p))))
    return q


def work(case):
    kind = case["kind"]
    if kind == "auxiliary":
        plan, parameters, aux = _auxiliary(case, 1)
        n, m = plan.orbital.nao(), plan.auxiliary.nao()
        bas = pack(plan.combined, type(parameters)(parameters.exponents + aux.exponents,
                                                   parameters.coefficients + aux.coefficients,
                                                   np.concatenate([parameters.centers, aux.centers]),
                                                   parameters.nuclear_coords))[1]
        o, x = bas[:plan.split], bas[plan.split:]
        flops = 0.0
        for r in x:
            for i, a in enumerate(o):
                for b in o[:i + 1]:
                    lt = int(a[1] + b[1] + r[1])
                    nr = lt // 2 + 1
                    nf = math.prod((l + 1) * (l + 2) // 2 for l in (int(a[1]), int(b[1]), int(r[1])))
                    flops += a[2] * b[2] * r[2] * (40 + 12 * nr + nr * (18 * (a[1] + b[1] + 1) * (r[1] + 1) + 3 * nf))
        return {"bytes": 8.0 * (m * m + m * n * (n + 1) // 2), "flops": float(flops)}
    tables = _tables(case, 1)
    if kind == "batch" and len(tables) > 8:
        scale, tables = len(tables) / 8.0, tables[:8]
    else:
        scale = 1.0
    data = flops = 0.0
    for t in tables:
        n = int(ao_offsets(t[1], case["cart"])[-1])
        nn = 8.0 * n * n
        if kind == "core":
            pairs = sum(int(a[2]) * int(b[2]) for i, a in enumerate(t[1]) for b in t[1][:i + 1])
            nuclei = int(np.count_nonzero(t[0][:, 0]))
            data += 5 * nn
            flops += pairs * nuclei * 400.0
            continue
        w = roofline.build_work(t[1], _schwarz(t) if case["cutoff"] else None, case["cutoff"], case["cart"])["total"]
        # derivatives of every centre (or parameter) take about four integrals' work
        flops += w["flop_eval"] * (0.0 if kind == "incore" else 4.0 if kind in ("geometry", "basis") else 1.0)
        flops += w["flop_dig"] * case["nb"] * (1 if case["symmetric"] else 2)
        data += nn * case["nb"] * (1 + case["with_j"] + case["with_k"])
        if kind == "incore":
            data += 8.0 * w["unique_ao_quartets"]
        if kind == "packed":
            data += 2 * 8.0 * w["unique_ao_quartets"]
        if kind == "fresh":
            data += 3 * nn
    return {"bytes": data * scale, "flops": flops * scale}


# ---------------------------------------------------------------------------
# the same values by plain 64-bit torch (McMurchie-Davidson over Hermite Gaussians)
# ---------------------------------------------------------------------------
_EXACT_AO = 200     # Cartesian AOs of the four-index tensor at most
_EXACT_AO_AD = 126  # with derivatives


class _Boys(torch.autograd.Function):
    """F_0..F_m(x) stacked on the first axis; dF_k/dx = -F_{k+1}."""

    @staticmethod
    def forward(ctx, x, m):
        top = m + 1
        small = x < 36.0
        xs = torch.where(small, x, torch.ones_like(x))
        e = torch.exp(-xs)
        term = torch.full_like(x, 1.0 / (2 * top + 1))
        total = term.clone()
        for k in range(1, 160):
            term = term * (2.0 * xs / (2 * (top + k) + 1))
            total = total + term
        f = [None] * (top + 1)
        f[top] = e * total
        for k in range(top - 1, -1, -1):
            f[k] = (2.0 * xs * f[k + 1] + e) / (2 * k + 1)
        xl = torch.where(small, torch.full_like(x, 36.0), x)
        el = torch.exp(-xl)
        g = 0.5 * torch.sqrt(math.pi / xl) * torch.erf(torch.sqrt(xl))
        for k in range(top + 1):
            f[k] = torch.where(small, f[k], g)
            g = ((2 * k + 1) * g - el) / (2.0 * xl)
        out = torch.stack(f)
        ctx.save_for_backward(out)
        return out[:m + 1]

    @staticmethod
    def backward(ctx, grad):
        (out,) = ctx.saved_tensors
        return -(grad * out[1:grad.shape[0] + 1]).sum(0), None


def _components(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _hermites(l):
    return [(t, u, v) for t in range(l + 1) for u in range(l + 1 - t) for v in range(l + 1 - t - u)]


def _expansion(la, lb, p, pa, pb):
    """1D Hermite coefficients E[i][j][t] (without the Gaussian prefactor)."""
    h = 0.5 / p
    e = {(0, 0): [torch.ones_like(p)]}

    def raise_(prev, shift):
        n = len(prev)
        out = []
        for t in range(n + 1):
            v = torch.zeros_like(p)
            if t > 0:
                v = v + h * prev[t - 1]
            if t < n:
                v = v + shift * prev[t]
            if t + 1 < n:
                v = v + (t + 1) * prev[t + 1]
            out.append(v)
        return out

    for i in range(la + 1):
        if i:
            e[i, 0] = raise_(e[i - 1, 0], pa)
        for j in range(1, lb + 1):
            e[i, j] = raise_(e[i, j - 1], pb)
    return e


def _coulomb(l, alpha, r):
    """R_tuv(alpha, r) for t + u + v <= l, stacked on the last axis in _hermites order."""
    f = _Boys.apply(alpha * (r * r).sum(-1), l)
    level = {}
    scale = torch.ones_like(alpha)
    for m in range(l + 1):
        level[m, (0, 0, 0)] = scale * f[m]
        scale = scale * (-2.0 * alpha)

    def get(m, k):
        if (m, k) not in level:
            axis = next(x for x in range(3) if k[x])
            k1 = tuple(v - (x == axis) for x, v in enumerate(k))
            v = r[..., axis] * get(m + 1, k1)
            if k1[axis]:
                k2 = tuple(v2 - (x == axis) for x, v2 in enumerate(k1))
                v = v + k1[axis] * get(m + 1, k2)
            level[m, k] = v
        return level[m, k]

    return torch.stack([get(0, k) for k in _hermites(l)], dim=-1)


class _Shells:
    """Contraction columns of the tables as Cartesian shells over the env tensor."""

    def __init__(self, atm, bas, env):
        self.atm, self.env = atm, env
        self.rows = []
        ao = 0
        for r in bas:
            for c in range(int(r[3])):
                self.rows.append((int(r[1]), int(r[2]), int(r[5]), int(r[6]) + c * int(r[2]), int(atm[r[0], 1]), ao))
                ao += (int(r[1]) + 1) * (int(r[1]) + 2) // 2
        self.n = ao

    def pairs(self, chosen, unit=False):
        """Primitive pairs of the shell pairs `chosen` (one class): with unit, the second
        function of every pair is the constant one."""
        dev = self.env.device
        la, lb = self.rows[chosen[0][0]][0], (0 if unit else self.rows[chosen[0][1]][0])
        cols = []
        for k, (i, j) in enumerate(chosen):
            _, na, ea, ca, ra, _ = self.rows[i]
            _, nb, eb, cb, rb, _ = (0, 1, 0, 0, ra, 0) if unit else self.rows[j]
            x, y = np.meshgrid(np.arange(na), np.arange(nb), indexing="ij")
            x, y = x.reshape(-1), y.reshape(-1)
            cols.append(np.stack([np.full(len(x), k), ea + x, ca + x, eb + y, cb + y, np.full(len(x), ra),
                                  np.full(len(x), rb)]))
        t = torch.as_tensor(np.concatenate(cols, axis=1), device=dev)
        factor = {0: 0.5 / math.sqrt(math.pi), 1: math.sqrt(3.0 / (4.0 * math.pi))}
        env = self.env
        a = env[t[1]]
        b = torch.zeros_like(a) if unit else env[t[3]]
        c = env[t[2]] * factor.get(la, 1.0)
        if not unit:
            c = c * env[t[4]] * factor.get(lb, 1.0)
        ra = torch.stack([env[t[5] + x] for x in range(3)], -1)
        rb = torch.stack([env[t[6] + x] for x in range(3)], -1)
        p = a + b
        centre = (a[:, None] * ra + b[:, None] * rb) / p[:, None]
        k = c * torch.exp(-a * b / p * ((ra - rb) ** 2).sum(-1))
        return dict(la=la, lb=lb, owner=t[0], count=len(chosen), p=p, b=b, centre=centre, k=k, ra=ra, rb=rb)

    def hermite(self, s, raised=0):
        """Hermite coefficients [primitive pair][component pair][tuv] of one class."""
        la, lb = s["la"], s["lb"]
        e = [_expansion(la, lb + raised, s["p"], s["centre"][:, x] - s["ra"][:, x], s["centre"][:, x] - s["rb"][:, x])
             for x in range(3)]
        if raised:
            return e
        zero = torch.zeros_like(s["p"])
        out = []
        for ca in _components(la):
            for cb in _components(lb):
                one = [e[x][ca[x], cb[x]] for x in range(3)]
                out.append(torch.stack([s["k"] * one[0][t] * one[1][u] * one[2][v]
                                        if t < len(one[0]) and u < len(one[1]) and v < len(one[2]) else zero
                                        for t, u, v in _hermites(la + lb)], -1))
        return torch.stack(out, 1)

    def classes(self, first=0, last=None):
        """Shell pairs i >= j of [first, last), grouped by class, higher momentum first."""
        groups = {}
        for i in range(first, len(self.rows) if last is None else last):
            for j in range(first, i + 1):
                a, b = (i, j) if self.rows[i][0] >= self.rows[j][0] else (j, i)
                groups.setdefault((self.rows[a][0], self.rows[b][0]), []).append((a, b))
        return groups

    def aos(self, chosen, which):
        l = self.rows[chosen[0][which]][0]
        w = (l + 1) * (l + 2) // 2
        return torch.as_tensor([[self.rows[p[which]][5] + c for c in range(w)] for p in chosen], device=self.env.device)


def _repulsion(s, es, t, et):
    """Contracted blocks [bra pair][ket pair][bra components][ket components], a bra
    range of pairs at a time: yields (first bra pair, blocks)."""
    lb, lk = s["la"] + s["lb"], t["la"] + t["lb"]
    hb, hk, ha = _hermites(lb), _hermites(lk), _hermites(lb + lk)
    where = {h: i for i, h in enumerate(ha)}
    pick = torch.as_tensor([[where[tuple(x + y for x, y in zip(p, q))] for q in hk] for p in hb], device=s["p"].device)
    sign = torch.as_tensor([(-1.0) ** sum(q) for q in hk], dtype=torch.float64, device=s["p"].device)
    room = max(1, int(4e7 / (len(t["p"]) * (len(hb) * len(hk) + 2 * len(ha)))))
    owner = s["owner"].cpu().numpy()
    begin = 0
    while begin < s["count"]:
        lo = int(np.searchsorted(owner, begin))
        end = begin + 1
        while end < s["count"] and np.searchsorted(owner, end + 1) - lo <= room:
            end += 1
        hi = int(np.searchsorted(owner, end))
        p, q = s["p"][lo:hi, None], t["p"][None]
        r = _coulomb(lb + lk, p * q / (p + q), s["centre"][lo:hi, None] - t["centre"][None])
        r = r * (2.0 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q)))[..., None]
        r = r[..., pick.reshape(-1)].reshape(hi - lo, len(t["p"]), len(hb), len(hk)) * sign
        x = torch.matmul(es[lo:hi, None], torch.matmul(r, et.transpose(1, 2)[None]))
        ket = torch.zeros((hi - lo, t["count"]) + x.shape[2:], dtype=x.dtype, device=x.device).index_add(1, t["owner"], x)
        out = torch.zeros((end - begin,) + ket.shape[1:], dtype=x.dtype, device=x.device)
        yield begin, out.index_add(0, s["owner"][lo:hi] - begin, ket)
        begin = end


def _eri(shells, visit):
    """Calls visit(a, b, c, d, block) for every block (ab|cd) of pair classes, AO index
    tensors [pairs][components] and block [bra][ket][a][b][c][d]; every ordered pair of
    shell pairs once, bra and ket each with i >= j."""
    groups = shells.classes()
    data = {k: (lambda s: (s, shells.hermite(s)))(shells.pairs(v)) for k, v in groups.items()}
    for kb, vb in groups.items():
        for kk, vk in groups.items():
            a, b, c, d = shells.aos(vb, 0), shells.aos(vb, 1), shells.aos(vk, 0), shells.aos(vk, 1)
            for first, x in _repulsion(*data[kb], *data[kk]):
                m = x.shape[0]
                x = x.reshape(m, x.shape[1], a.shape[1], b.shape[1], c.shape[1], d.shape[1])
                visit(a[first:first + m], b[first:first + m], c, d, x)


def _eri_tensor(shells):
    out = torch.zeros((shells.n,) * 4, dtype=torch.float64, device=shells.env.device)

    def visit(a, b, c, d, x):
        a, b = a[:, None, :, None, None, None], b[:, None, None, :, None, None]
        c, d = c[None, :, None, None, :, None], d[None, :, None, None, None, :]
        for p, q in ((a, b), (b, a)):
            for r, s in ((c, d), (d, c)):
                out[p, q, r, s] = x

    _eri(shells, visit)
    return out


def _solid(l):
    """Cartesian components -> real solid harmonics of libcint's convention (rows m = -l..l;
    identity for s and p), from the closed form of Helgaker, Jorgensen and Olsen."""
    comp = _components(l)
    if l < 2:
        return np.eye(len(comp))
    out = np.zeros((2 * l + 1, len(comp)))
    for m in range(-l, l + 1):
        am, half = abs(m), int(m < 0)
        norm = math.sqrt(2.0 * math.factorial(l + am) * math.factorial(l - am) / (2.0 if m == 0 else 1.0))
        norm *= math.sqrt((2 * l + 1) / (4 * math.pi)) / (2 ** am * math.factorial(l))
        for t in range((l - am) // 2 + 1):
            for u in range(t + 1):
                for v in range(half, am + 1, 2):
                    c = (-1) ** (t + (v - half) // 2) * 0.25 ** t * math.comb(l, t) * math.comb(t, u) * math.comb(am, v)
                    c *= math.comb(l - t, am + t) if am + t <= l - t else 0
                    if c:
                        out[m + l, comp.index((2 * t + am - 2 * u - v, 2 * u + v, l - 2 * t - am))] += norm * c
    return out


def _transform(bas, cart, dev):
    rows = [np.eye((int(r[1]) + 1) * (int(r[1]) + 2) // 2) if cart else _solid(int(r[1])) for r in bas for _ in range(r[3])]
    out = np.zeros((sum(x.shape[0] for x in rows), sum(x.shape[1] for x in rows)))
    i = j = 0
    for x in rows:
        out[i:i + x.shape[0], j:j + x.shape[1]] = x
        i, j = i + x.shape[0], j + x.shape[1]
    return torch.as_tensor(out, device=dev)


def _exact_jk(table, cart, dens):
    """J and K of (nb, n, n) densities, and the four-index tensor in the AO basis."""
    atm, bas, env = table
    dev = dens.device
    eri = _eri_tensor(_Shells(atm, bas, torch.as_tensor(env, device=dev)))
    t = _transform(bas, cart, dev)
    if not cart:
        for _ in range(4):
            eri = torch.tensordot(eri, t, dims=([0], [1]))
    n = t.shape[0]
    flat = dens.reshape(-1, n * n)
    j = (flat @ eri.reshape(n * n, n * n)).reshape(dens.shape)
    k = (flat @ eri.transpose(1, 2).reshape(n * n, n * n)).reshape(dens.shape)
    return j, k, eri


def _exact_gradient(table, cart, d, cj, ck):
    """d/d env of sum(cj J(d)) + sum(ck K(d)), by autograd over the Hermite integrals."""
    atm, bas, env = table
    env = torch.as_tensor(env, device=d.device).requires_grad_(True)
    t = _transform(bas, cart, d.device)
    up = lambda x: torch.zeros((t.shape[1],) * 2, dtype=x.dtype, device=x.device) if x is None else t.T @ x @ t  # noqa: E731
    dc, jc, kc = up(d), up(cj if cj is not None else 0 * d), up(ck if ck is not None else 0 * d)
    total = torch.zeros_like(env)
    shells = _Shells(atm, bas, env)
    groups = shells.classes()
    for vb in groups.values():
        for vk in groups.values():
            a, b, c, e = shells.aos(vb, 0), shells.aos(vb, 1), shells.aos(vk, 0), shells.aos(vk, 1)
            # the Hermite data is rebuilt per block so that each block's graph is freed
            at = 0
            while at < len(vb):
                part = vb[at:at + 48]
                s, u = shells.pairs(part), shells.pairs(vk)
                value = 0.0
                for first, x in _repulsion(s, shells.hermite(s), u, shells.hermite(u)):
                    m = x.shape[0]
                    x = x.reshape(m, x.shape[1], a.shape[1], b.shape[1], c.shape[1], e.shape[1])
                    lo = at + first
                    ia, ib = a[lo:lo + m][:, None, :, None, None, None], b[lo:lo + m][:, None, None, :, None, None]
                    ic, ie = c[None, :, None, None, :, None], e[None, :, None, None, None, :]
                    w = 0.0
                    bra = [(ia, ib, 1.0), (ib, ia, torch.as_tensor([i != j for i, j in part[first:first + m]]).to(x))]
                    ket = [(ic, ie, 1.0), (ie, ic, torch.as_tensor([i != j for i, j in vk]).to(x))]
                    for p, q, f in bra:
                        f = f if isinstance(f, float) else f[:, None, None, None, None, None]
                        for r, v, g in ket:
                            g = g if isinstance(g, float) else g[None, :, None, None, None, None]
                            w = w + f * g * (jc[p, q] * dc[r, v] + kc[p, r] * dc[q, v])
                    value = value + (w * x).sum()
                total += torch.autograd.grad(value, env)[0]
                at += len(part)
    return total


def _exact_core(table, cart, d, w):
    """S, T, V and the one-electron gradient rows, sum d d(T + V)/dR - w dS/dR."""
    atm, bas, env = table
    env = torch.as_tensor(env, device=d.device).requires_grad_(True)
    shells = _Shells(atm, bas, env)
    t = _transform(bas, cart, d.device)
    dc, wc = t.T @ d @ t, t.T @ w @ t
    nuclei = [int(i) for i in np.flatnonzero(atm[:, 0])]
    charge = torch.as_tensor(atm[nuclei, 0].astype(np.float64), device=d.device)
    mats = [torch.zeros((shells.n, shells.n), dtype=torch.float64, device=d.device) for _ in range(3)]
    total = torch.zeros_like(env)
    for chosen in shells.classes().values():
        s = shells.pairs(chosen)
        la, lb, p = s["la"], s["lb"], s["p"]
        e = shells.hermite(s, raised=2)
        full = shells.hermite(s)
        where = torch.stack([torch.stack([env[int(atm[i, 1]) + x] for x in range(3)]) for i in nuclei])
        r = _coulomb(la + lb, p[:, None].expand(-1, len(nuclei)), s["centre"][:, None] - where[None])
        r = -(r * charge[None, :, None]).sum(1) * (2.0 * math.pi / p)[:, None]
        ov = s["k"] * (math.pi / p) ** 1.5
        blocks = [[], [], torch.matmul(full, r[:, :, None])[..., 0]]
        for ca in _components(la):
            for cb in _components(lb):
                o = [e[x][ca[x], cb[x]][0] for x in range(3)]
                k = []
                for x in range(3):
                    v = -2.0 * s["b"] ** 2 * e[x][ca[x], cb[x] + 2][0] + s["b"] * (2 * cb[x] + 1) * o[x]
                    if cb[x] > 1:
                        v = v - 0.5 * cb[x] * (cb[x] - 1) * e[x][ca[x], cb[x] - 2][0]
                    k.append(v)
                blocks[0].append(ov * o[0] * o[1] * o[2])
                blocks[1].append(ov * (k[0] * o[1] * o[2] + o[0] * k[1] * o[2] + o[0] * o[1] * k[2]))
        blocks = [torch.stack(x, 1) if isinstance(x, list) else x for x in blocks]
        a, b = shells.aos(chosen, 0)[:, :, None], shells.aos(chosen, 1)[:, None, :]
        two = torch.as_tensor([1.0 if i == j else 2.0 for i, j in chosen], dtype=torch.float64, device=d.device)
        value = 0.0
        for x, m, weight in zip(blocks, mats, (-wc, dc, dc)):
            y = torch.zeros((len(chosen), x.shape[1]), dtype=x.dtype, device=x.device).index_add(0, s["owner"], x)
            y = y.reshape(len(chosen), a.shape[1], b.shape[2])
            m[a, b] = y.detach()
            m[b, a] = y.detach()
            value = value + (two[:, None, None] * 0.5 * (weight[a, b] + weight[b, a]) * y).sum()
        total += torch.autograd.grad(value, env)[0]
    rows = torch.stack([total[int(r[1]):int(r[1]) + 3] for r in atm])
    return tuple(t @ m @ t.T for m in mats) + (rows,)


def _exact_auxiliary(case, seed, dev):
    plan, parameters, aux = _auxiliary(case, seed)
    both = type(parameters)(parameters.exponents + aux.exponents, parameters.coefficients + aux.coefficients,
                            np.concatenate([parameters.centers, aux.centers]), parameters.nuclear_coords)
    atm, bas, env = pack(plan.combined, both)
    shells = _Shells(atm, bas, torch.as_tensor(env, device=dev))
    split = int(sum(bas[:plan.split, 3]))
    n_orb = shells.rows[split][5]
    m_aux = shells.n - n_orb
    groups = {}
    for i in range(split, len(shells.rows)):
        groups.setdefault(shells.rows[i][0], []).append((i, i))
    kets = [(v, (lambda s: (s, shells.hermite(s)))(shells.pairs(v, unit=True))) for v in groups.values()]
    two = torch.zeros((m_aux, m_aux), dtype=torch.float64, device=dev)
    three = torch.zeros((m_aux, n_orb, n_orb), dtype=torch.float64, device=dev)
    for vk, ket in kets:
        c = shells.aos(vk, 0) - n_orb
        for vb, bra in kets:
            a = shells.aos(vb, 0) - n_orb
            for first, x in _repulsion(*bra, *ket):
                two[a[first:first + len(x), None, :, None], c[None, :, None, :]] = x
        for vb in shells.classes(0, split).values():
            s = shells.pairs(vb)
            a, b = shells.aos(vb, 0), shells.aos(vb, 1)
            for first, x in _repulsion(s, shells.hermite(s), *ket):
                m = len(x)
                x = x.reshape(m, len(vk), a.shape[1], b.shape[1], c.shape[1])
                ia, ib = a[first:first + m, None, :, None, None], b[first:first + m, None, None, :, None]
                three[c[None, :, None, None, :], ia, ib] = x
                three[c[None, :, None, None, :], ib, ia] = x
    to, ta = _transform(bas[:plan.split], case["cart"], dev), _transform(bas[plan.split:], case["cart"], dev)
    two = ta @ two @ ta.T
    three = to @ (ta @ three.reshape(m_aux, -1)).reshape(-1, n_orb, n_orb) @ to.T
    i, j = np.tril_indices(three.shape[1])
    return two, three[:, torch.as_tensor(i, device=dev), torch.as_tensor(j, device=dev)]


def exact(case, seed):
    kind = case["kind"]
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if kind == "auxiliary":
        return _exact_auxiliary(case, seed, dev)
    tables = _tables(case, seed)
    dens = torch.as_tensor(_matrices(case, seed, tables)).to(dev)
    size = max(int(ao_offsets(t[1], True)[-1]) for t in tables)
    if kind == "core":
        w = torch.as_tensor(_matrix(tables[0], case["cart"], np.random.default_rng([seed, 8]))).to(dev)
        return _exact_core(tables[0], case["cart"], dens[0], w)
    if kind in ("geometry", "basis"):
        if size > _EXACT_AO_AD:
            return None
        g = _exact_gradient(tables[0], case["cart"], dens[0], *_cotangents(case, dens[0]))
        atm, bas, _ = tables[0]
        if kind == "geometry":
            return torch.stack([g[int(r[1]):int(r[1]) + 3] for r in atm])
        keep = torch.zeros_like(g)
        for r in bas:
            keep[int(r[5]):int(r[5] + r[2])] = 1.0
            keep[int(r[6]):int(r[6] + r[2] * r[3])] = 1.0
        return g * keep
    if kind == "batch" or size > _EXACT_AO:
        return None
    j, k, eri = _exact_jk(tables[0], case["cart"], dens)
    if kind == "packed":
        i, m = (torch.as_tensor(x, device=dev) for x in np.tril_indices(dens.shape[-1]))
        pair = eri[i, m][:, i, m]
        i, m = (torch.as_tensor(x, device=dev) for x in np.tril_indices(len(pair)))
        return pair[i, m], (j, k)
    if kind == "direct":
        zero = torch.zeros_like(j)
        return (j if case["with_j"] else zero), (k if case["with_k"] else zero)
    both = torch.stack([x for x, wanted in ((j, case["with_j"]), (k, case["with_k"])) if wanted])
    if kind == "fresh":
        zero = torch.zeros_like(dens[0])
        return _exact_core(tables[0], case["cart"], zero, zero)[:3], both
    return both
