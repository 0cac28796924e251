"""GPU: the allocation-free entry point captured into a HIP graph and replayed, and at its limit."""
import ctypes

import numpy as np
import pytest

from chronusq_public_amd import _lib
from chronusq_public_amd import basis as B
from chronusq_public_amd import molecule as M
from chronusq_public_amd.aointegrals import AOIntegrals, COULOMB, EXCHANGE

pytestmark = pytest.mark.gpu


def _context(m, basis):
    mol = M.water_cluster(m, seed=3, box_ang=M.scaled_box(m))
    ao = AOIntegrals(B.build_basis(basis, mol.Z, mol.coords_bohr))
    ao.thresholdSchwartz = 1e-12
    return ao


def _noalloc(ao, X, AX, types, scales):
    import torch
    n = len(X)
    xp = (ctypes.c_void_p * n)(*[t.data_ptr() for t in X])
    ap = (ctypes.c_void_p * n)(*[t.data_ptr() for t in AX])
    ty, sc = (ctypes.c_int * n)(*types), (ctypes.c_double * n)(*scales)
    _lib.check(_lib.load().cq_contract_direct_device_noalloc(ao._h, n, xp, ap, ty, sc, ao.nBasis, ao.nBasis,
                                                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), ao._h)


@pytest.mark.parametrize("m,basis", [(1, "6-31g*"), (4, "cc-pvdz")])
def test_captured_contraction_replays(m, basis):
    """Three replays with other densities, eager contractions and synchronisations between them, each
    against the eager result."""
    import torch
    print(f"[capture] {m} {basis}", flush=True)
    ao = _context(m, basis)
    N = ao.nBasis
    rng = np.random.default_rng(5)
    X = torch.zeros((N, N), dtype=torch.float64, device="cuda")
    J, K = torch.zeros_like(X), torch.zeros_like(X)
    types, scales = [COULOMB, EXCHANGE], [1.0, -0.5]

    def step():
        J.zero_()
        K.zero_()
        _noalloc(ao, [X, X], [J, K], types, scales)

    def density():
        A = rng.uniform(-1, 1, (N, N))
        X.copy_(torch.from_numpy(A + A.T))

    density()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(3):
        density()
        eager = [torch.zeros_like(X), torch.zeros_like(X)]
        ao.newTwoEContractDirect([X, X], eager, types, scales)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for got, want in zip((J, K), eager):
            assert want.abs().max().item() > 1.0
            assert (got - want).abs().max().item() < 1e-10


@pytest.mark.parametrize("m,densities", [(51, 1), (18, 8)])
def test_largest_calls_that_fit(m, densities):
    """Just below 5 ncart^2 doubles per density of 64 MiB (one water more is refused): the same as the
    allocating entry point."""
    import torch
    print(f"[capture] {m} waters, {densities} densities", flush=True)
    ao = _context(m, "cc-pvdz")
    room = 64 << 20
    assert densities * (40 * ao.nCart ** 2 + 4) <= room < densities * (40 * (ao.nCart + 25) ** 2 + 4)
    X, want, got = [], [], []
    for i in range(densities):
        d = torch.rand(ao.nBasis, dtype=torch.float64, generator=torch.Generator().manual_seed(i)).cuda()
        X.append(torch.diag(d) + 1e-3 * torch.outer(d, d))
        want.append(torch.zeros_like(X[i]))
        got.append(torch.zeros_like(X[i]))
    types, scales = [COULOMB, EXCHANGE][:1 + (densities > 1)] + [EXCHANGE] * max(0, densities - 2), [1.0] * densities
    ao.newTwoEContractDirect(X, want, types, scales)
    _noalloc(ao, X, got, types, scales)
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert w.abs().max().item() > 1e-3
        assert (g - w).abs().max().item() < 1e-10 * max(1.0, w.abs().max().item())
