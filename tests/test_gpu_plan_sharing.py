"""Calls on one plan that share no workspace: the allocation-free J/K build
beside the derivative calls.  A call issued on another stream while one of
them is under capture stays out of the graph, its result is that of a call
alone, and so are the graph's replays; calls from two threads at once give
what they give alone."""
import ctypes
import threading

import pytest

from gradscf_amd import molecule as M
from tests import systems

pytestmark = pytest.mark.gpu


class _Calls:
    def __init__(self):
        import torch
        from gradscf_amd.jk import DirectJKPlan
        _, _, *tables = systems.tables(M.water_cluster(2, seed=3, box=6.0), "cc-pvdz", cart=False)
        self.plan = DirectJKPlan(*tables, cart=False, cutoff=0.0)
        self.d = torch.as_tensor(systems.random_density(self.plan.nao, seed=8)[0], device="cuda").contiguous()
        self.out = torch.empty((2, 1, self.plan.nao, self.plan.nao), dtype=torch.float64, device="cuda")

    def build(self):
        import torch
        from gradscf_amd import _native
        _native.check(_native.lib().gscf_jk_build_noalloc(
            self.plan._handle, self.d.data_ptr(), 1, self.out.data_ptr(), 1, 1,
            _native.FLAG_SYMMETRIC_DENSITY | _native.FLAG_NO_VALIDATE, ctypes.c_double(0.0),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        return self.out

    def int1e_gradient(self):
        return self.plan.int1e_gradient(self.d, self.d)

    def jk_geometry_vjp(self):
        return self.plan.jk_geometry_vjp(self.d, self.d, self.d)

    def jk_param_vjp(self):
        return self.plan.jk_param_vjp(self.d, self.d, self.d)


def _same(got, ref):
    # sums of atomic adds in another order
    return float((got - ref).abs().max()) < 1e-12 * max(1.0, float(ref.abs().max()))


DERIVATIVES = ["int1e_gradient", "jk_geometry_vjp", "jk_param_vjp"]


@pytest.mark.parametrize("captured,eager", [("build", x) for x in DERIVATIVES] + [(x, "build") for x in DERIVATIVES])
def test_call_beside_a_capture(captured, eager):
    import torch
    calls = _Calls()
    captured, eager = getattr(calls, captured), getattr(calls, eager)
    ref_captured, ref_eager = captured().clone(), eager().clone()
    torch.cuda.synchronize()
    other, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        held = captured()
        with torch.cuda.stream(other):
            got = eager()
    other.synchronize()
    assert _same(got, ref_eager)
    for _ in range(3):
        held.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        with torch.cuda.stream(other):
            again = eager()
        torch.cuda.synchronize()
        assert _same(held, ref_captured) and _same(again, ref_eager)


@pytest.mark.parametrize("name", DERIVATIVES)
def test_calls_on_two_threads(name):
    import torch
    calls = _Calls()
    refs = {n: getattr(calls, n)().clone() for n in ("build", name)}
    torch.cuda.synchronize()
    bad = []

    def work(n):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(50):
                    got = getattr(calls, n)()
                    torch.cuda.current_stream().synchronize()
                    if not _same(got, refs[n]):
                        bad.append(n)
        except Exception as e:  # noqa: BLE001 (reported by the main thread)
            bad.append(e)

    threads = [threading.Thread(target=work, args=(n,)) for n in refs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
