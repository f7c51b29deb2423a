"""Packed J/K of few AOs (one launch, sums in one thread) at the edges of its
range, for both layouts and every operator selection, on v(ab, cd) = x_ab x_cd,
whose J and K are X (X . D) and X D X."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 11, 12, 13])
@pytest.mark.parametrize("ndim", [1, 2])
@pytest.mark.parametrize("with_j,with_k", [(1, 1), (1, 0), (0, 1)])
def test_small_packed_jk(n, ndim, with_j, with_k):
    import torch
    from gradscf_amd import _native
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n * (n + 1) // 2, dtype=torch.float64, device="cuda", generator=g)
    x[len(x) // 2] = 0.0
    i, j = torch.tril_indices(n, n, device="cuda")
    full = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    full[i, j] = full[j, i] = x
    pairs = x[:, None] * x[None, :]
    if ndim == 1:
        p, q = torch.tril_indices(len(x), len(x), device="cuda")
        eri = pairs[p, q].contiguous()
    else:
        # only the lower triangle is read
        eri = (pairs.tril() + torch.full_like(pairs, 7.0).triu(1)).contiguous()
    d = torch.randn((5, n, n), dtype=torch.float64, device="cuda", generator=g)
    out = torch.full((with_j + with_k, 5, n, n), float("nan"), dtype=torch.float64, device="cuda")
    _native.check(_native.lib().gscf_packed_jk(eri.data_ptr(), eri.numel(), ndim, d.data_ptr(), 5, n, out.data_ptr(),
                                               with_j, with_k,
                                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    for b in range(5):
        # rounding: n^2 additions of terms whose absolute values sum to top
        if with_j:
            top = full.abs() * (full.abs() * d[b].abs()).sum()
            assert bool(((out[0, b] - full * (full * d[b]).sum()).abs() <= 1e-13 * top).all())
            assert torch.equal(out[0, b], out[0, b].T)
        if with_k:
            top = full.abs() @ d[b].abs() @ full.abs()
            assert bool(((out[-1, b] - full @ d[b] @ full).abs() <= 1e-13 * top).all())
