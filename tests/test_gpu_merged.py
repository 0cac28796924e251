"""GPU: the class pairs of a call in a few merged launches (the default of an FP64 call) against the
oracle and against a launch per class pair, where the two can differ: one and two shells, class
pairs without a partner class, the three sizes of primitive blocks, both keyed sides, open shell, a
non-symmetric density, class pairs of both kinds in one call, task lists in several batches, and
several molecules; and the one-electron kernel at the edges of its 64-pair workgroups.  (The shipped
bases hold d as pure shells: Cartesian ones are in test_gpu_shell_forms.py.)"""
import numpy as np
import pytest

import oracle
from chronusq_public_amd import _lib
from chronusq_public_amd import basis as B
from chronusq_public_amd import molecule as M
from chronusq_public_amd.aointegrals import AOIntegrals, COULOMB, EXCHANGE

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _atoms(*zs):
    return M.Molecule(np.array(zs), np.array([[0.3 * i, -0.2 * i, 1.9 * i] for i in range(len(zs))]))


def _water(m):
    return M.water_cluster(m, seed=5, box_ang=M.scaled_box(m))


SYSTEMS = {
    "H/6-31g": (lambda: _atoms(1), "6-31g"),            # (ss|ss) alone
    "Ne/6-31g": (lambda: _atoms(10), "6-31g"),          # no d class
    "NeH/cc-pvdz": (lambda: _atoms(10, 1), "cc-pvdz"),  # every class, few pairs
    "H2O 4/6-31g": (lambda: _water(4), "6-31g"),        # more than 300 pairs, (ss) the ket of (pp)
    "H2O 4/cc-pvdz": (lambda: _water(4), "cc-pvdz"),
    "H2O 9/6-31g": (lambda: _water(9), "6-31g"),        # 117 functions, several groups a class
}


def _build(name):
    make, basis = SYSTEMS[name]
    mol = make()
    return mol, B.build_basis(basis, mol.Z, mol.coords_bohr)


def _matrices(N, seed, symmetric=True):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(2):
        X = rng.uniform(-1, 1, (N, N))
        out.append(np.asfortranarray(0.5 * (X + X.T) if symmetric else X))
    return out


def _contract(ao, Xs, types, scales):
    ao.thresholdSchwartz = 1e-12
    AX = [np.zeros((ao.nBasis, ao.nBasis), order="F") for _ in Xs]
    ao.newTwoEContract(Xs, AX, types, scales)
    return AX, sum(ao.quartet_counts().values())


@pytest.mark.parametrize("name", list(SYSTEMS))
@pytest.mark.parametrize("symmetric", [True, False])
def test_merged_launches_match_oracle_and_separate_launches(name, symmetric):
    print(f"[merged] {name} symmetric={symmetric}", flush=True)
    L = _lib.load()
    _, bs = _build(name)
    ob = oracle.OracleBasis(bs)
    A, C = _matrices(bs.nbasis, 31, symmetric)
    Xs, types, scales = [A, A, C], [COULOMB, EXCHANGE, EXCHANGE], [1.0, -0.5, 0.25]
    ao = AOIntegrals(bs)
    Q = ao.computeSchwartz()
    want = [np.zeros((ob.nbf, ob.nbf), order="F") for _ in Xs]
    n = ob.contract_direct(Q, 1e-12, Xs, want, [0, 1, 1], scales)

    def check(what):
        print(f"[merged]   {what}", flush=True)
        got, m = _contract(ao, Xs, types, scales)
        assert m == n, what
        for g, w in zip(got, want):
            assert np.abs(g - w).max() < TOL, what

    check("merged")
    check("merged again")
    _lib.check(L.cq_set_launch_streams(ao._h, 1), ao._h)
    check("a launch per class pair")
    _lib.check(L.cq_set_launch_streams(ao._h, 4), ao._h)
    for k in range(0, L.cq_num_class_pairs(), 3):   # every third class pair leaves the merged launches
        _lib.check(L.cq_set_class_digestion(ao._h, k, (2, 0, 1)[k // 3 % 3]), ao._h)
    check("both kinds in one call")
    for k in range(0, L.cq_num_class_pairs(), 3):
        _lib.check(L.cq_set_class_digestion(ao._h, k, -1), ao._h)
    entries, _ = ao.task_plan()
    ao.set_task_budget(max(1, entries // 40))
    check("the large class pairs in several batches")


def test_merged_launches_several_molecules():
    """Every block of a batched context is that molecule's own J and K; class pairs that only some
    molecules have."""
    names = ["H/6-31g", "Ne/6-31g", "H2O 4/6-31g"]
    bases = [_build(n)[1] for n in names]
    big = AOIntegrals.batch(bases)
    N = big.nBasis
    X = np.zeros((N, N), order="F")
    off = 0
    for i, b in enumerate(bases):
        X[off:off + b.nbasis, off:off + b.nbasis] = _matrices(b.nbasis, 60 + i)[0]
        off += b.nbasis
    (J, K), _ = _contract(big, [X, X], [COULOMB, EXCHANGE], [1.0, -0.5])
    off = 0
    for b in bases:
        sl = slice(off, off + b.nbasis)
        off += b.nbasis
        ob = oracle.OracleBasis(b)
        want = [np.zeros((ob.nbf, ob.nbf), order="F") for _ in range(2)]
        x = np.asfortranarray(X[sl, sl])
        ob.contract_direct(AOIntegrals(b).computeSchwartz(), 1e-12, [x, x], want, [0, 1], [1.0, -0.5])
        assert np.abs(J[sl, sl] - want[0]).max() < TOL and np.abs(K[sl, sl] - want[1]).max() < TOL


@pytest.mark.parametrize("name", list(SYSTEMS))
def test_one_electron_workgroup_edges(name):
    """One pair, a few pairs of one class, more nuclei than wavefronts, several workgroups a class:
    S, T and V against the oracle (1e-10, as for the larger systems)."""
    mol, bs = _build(name)
    got = AOIntegrals(bs).computeAOOneE(mol)
    for g, w in zip(got, oracle.OracleBasis(bs).one_electron(mol)):
        g = g.cpu().numpy()
        assert np.isfinite(g).all() and np.abs(g - w).max() < TOL * max(1.0, np.abs(w).max())


@pytest.mark.parametrize("name,basis", [("H/6-31g", None), ("NeH/cc-pvdz", None), ("NeH/cc-pvdz", "6-31g*"),
                                        ("H2O 4/cc-pvdz", None), ("H2O 4/cc-pvdz", "6-31g*")])
def test_schwarz_bounds_lane_groups(name, basis):
    """Schwarz bounds with 1 to 64 lanes per pair, pure and Cartesian d, one pair and many per class,
    against the oracle to 1e-12 of the largest."""
    mol, bs = _build(name)
    if basis:
        bs = B.build_basis(basis, mol.Z, mol.coords_bohr)
    Q, want = AOIntegrals(bs).computeSchwartz(), oracle.OracleBasis(bs).schwarz()
    assert np.abs(Q - Q.T).max() == 0.0
    assert np.abs(Q - want).max() <= 1e-12 * max(1.0, want.max())


@pytest.mark.parametrize("name,basis,m", [("more than 6000 pairs", "cc-pvdz", 11), ("up to 6000", "6-31g*", 8)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_merged_launches_by_primitive_blocks(name, basis, m, symmetric):
    """On either side of the line to the largest primitive blocks (the merged launches then share the
    orders and block counts of the launches per class pair): two densities in merged launches, a launch per
    class pair, and with the large class pairs in several batches beside merged ones."""
    print(f"[merged] {name} symmetric={symmetric}", flush=True)
    L = _lib.load()
    mol = _water(m)
    bs = B.build_basis(basis, mol.Z, mol.coords_bohr)
    ao = AOIntegrals(bs)
    assert (ao.nShellPair > 6000) == (m == 11)
    A, C = _matrices(bs.nbasis, 41, symmetric)
    Xs, types, scales = [A, A, C], [COULOMB, EXCHANGE, EXCHANGE], [1.0, -0.5, 0.25]
    _lib.check(L.cq_set_launch_streams(ao._h, 1), ao._h)
    want, n = _contract(ao, Xs, types, scales)
    _lib.check(L.cq_set_launch_streams(ao._h, 4), ao._h)
    entries, batches = ao.task_plan()
    assert batches == 1 and n > 0
    for budget in (None, entries // 40):
        if budget:
            ao.set_task_budget(budget)
            assert ao.task_plan()[1] > 1
        got, k = _contract(ao, Xs, types, scales)
        assert k == n
        for g, w in zip(got, want):
            assert np.abs(g - w).max() < TOL
