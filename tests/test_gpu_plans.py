"""GPU: what a context reports of its plans and what it reserves for them -- the work sums of a call in
merged launches, and the task plan."""
import ctypes

import numpy as np
import pytest

from chronusq_public_amd import _lib
from chronusq_public_amd import basis as B
from chronusq_public_amd import molecule as M
from chronusq_public_amd.aointegrals import AOIntegrals, COULOMB, EXCHANGE

pytestmark = pytest.mark.gpu


def _water(m, basis):
    mol = M.water_cluster(m, seed=5, box_ang=M.scaled_box(m))
    return B.build_basis(basis, mol.Z, mol.coords_bohr)


def _density(N, seed=2):
    X = np.random.default_rng(seed).uniform(-1, 1, (N, N))
    return np.asfortranarray(0.5 * (X + X.T))


def _contract(ao, X):
    AX = [np.zeros((ao.nBasis, ao.nBasis), order="F") for _ in range(2)]
    ao.newTwoEContract([X, X], AX, [COULOMB, EXCHANGE], [1.0, -0.5])
    return AX


@pytest.mark.parametrize("m,basis", [(1, "6-31g*"), (2, "cc-pvdz"), (6, "6-31g")])
def test_work_sums_do_not_depend_on_the_launches(m, basis):
    """Primitive quartets, K_ab, transform operations and integrals of a call in merged launches (with
    primitive blocks and orientations of their own) are those of a launch per class pair."""
    print(f"[plans] work sums {m} {basis}", flush=True)
    L = _lib.load()
    nc = L.cq_num_class_pairs()
    bs = _water(m, basis)
    ao = AOIntegrals(bs)
    ao.thresholdSchwartz = 1e-12
    X = _density(bs.nbasis)
    sums = []
    for streams in (4, 1):
        _lib.check(L.cq_set_launch_streams(ao._h, streams), ao._h)
        _contract(ao, X)
        w = (ctypes.c_double * (4 * nc))()
        _lib.check(L.cq_get_work_stats(ao._h, w, nc), ao._h)
        sums.append(np.array(w).reshape(nc, 4))
    assert sums[0][:, 0].sum() > 0
    assert np.array_equal(sums[0], sums[1])


def test_plans_that_no_launch_uses_reserve_nothing():
    """(H2O)100/cc-pVDZ: the merged tiles of class pairs with many d or p rows do not fit the LDS, and
    the largest class pairs take several batches; neither plan may size the buffers.  Beside the task
    lists (8 B per entry) a context holds their segments (16 B per region of at least 64 swept pairs'
    entries and a header), the pair tables and matrices over shells: less than a twentieth of the lists."""
    import torch
    bs = _water(100, "cc-pvdz")
    AOIntegrals(_water(1, "cc-pvdz")).close()   # the library's own first allocations
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    ao = AOIntegrals(bs)
    used = free - torch.cuda.mem_get_info()[0]
    entries, batches = ao.task_plan()
    ao.close()
    print(f"[plans] context {used / 2**30:.2f} GiB, task lists {entries * 8 / 2**30:.2f} GiB, {batches} batches", flush=True)
    assert batches > 1
    assert used - 8 * entries < 8 * entries / 20


@pytest.mark.parametrize("m,tile", [(4, (4, 256)), (24, (16, 512))])
def test_own_launches_keep_their_tiles(m, tile):
    """A class pair's own launch has rows of its own up to 20000 shell pairs (many small items), the
    merged launches' rows above: (ss|ds) of (H2O)4 and (H2O)24 in cc-pVDZ, on either side of the line."""
    L = _lib.load()
    ls = [ctypes.c_int() for _ in range(4)]
    ssds = None
    for k in range(L.cq_num_class_pairs()):
        L.cq_class_pair_info(k, *[ctypes.byref(x) for x in ls])
        if [x.value for x in ls] == [0, 0, 2, 0]:
            ssds = k
    ao = AOIntegrals(_water(m, "cc-pvdz"))
    assert (ao.nShellPair > 20000) == (m == 24)
    assert ao.class_tile(ssds)[:2] == tile


def test_workspace_of_a_contraction():
    """What the first contraction of eight densities adds to a context (the least of four equal ones: the
    runtime's own first allocations for the kernels come on top in the first): per density three
    matrices of accumulators, the density and its transpose, and two lists in pair order of at most half
    a matrix each (njel <= (ncart^2 + 6 ncart) / 2 elements), and 4 MiB for the flags and the pages."""
    import torch
    bs = _water(40, "cc-pvdz")
    used = []
    for _ in range(4):
        ao = AOIntegrals(bs)
        ao.thresholdSchwartz = 1e-12
        nc = ao.nCart
        X = [torch.zeros((ao.nBasis, ao.nBasis), dtype=torch.float64, device="cuda").fill_diagonal_(1.0 + i) for i in range(8)]
        AX = [torch.zeros_like(x) for x in X]
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        ao.newTwoEContractDirect(X, AX, [EXCHANGE] * 8, [-0.5] * 8)
        torch.cuda.synchronize()
        used.append(free - torch.cuda.mem_get_info()[0])
        ao.close()
    print(f"[plans] workspace {min(used) / 2**20:.1f} MiB, {min(used) / (8 * 8 * nc * nc):.2f} matrices a density", flush=True)
    assert 0 < min(used) <= 8 * 8 * (6 * nc * nc + 6 * nc) + (4 << 20)
