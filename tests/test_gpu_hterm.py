"""H|psi> and transforms of the Smolyak terms in register blocks against the
oracle: every group shape of the kernel and the generic one (the 1D laws 1 + 2l functions on
2 + 2l or 1 + 2l points, 1 + l on 2 + l, 2 + 2l on 3 + 2l; slots up to 19
functions), terms of one function, terms whose V part runs in slabs (seven
active modes), one to nine vectors, the kinetic part with and without a
q-linear G and off-diagonal terms, and a G(q) that is not symmetric in its two
indices, which the older term kernels keep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL64 = 1e-12  # the parity bar of every FP64 H|psi> test

CASES = [(1, 3, (1, 2, 2, 2), 10, "ga", 1), (2, 9, (1, 2, 2, 2), 10, "ga", 1), (3, 6, (1, 2, 2, 2), 10, "ga", 4),
         (4, 4, (1, 2, 2, 2), 10, "ga", 3), (4, 4, (1, 2, 1, 2), 10, "ga", 1), (4, 3, (1, 1, 2, 1), 10, "ga", 2),
         (3, 3, (2, 2, 3, 2), 10, "ga", 9), (6, 5, (1, 2, 2, 2), 10, "ga", 2), (6, 4, (1, 2, 2, 2), 10, "ga", 7),
         (4, 4, (1, 2, 2, 2), 10, "g0", 3), (4, 4, (1, 2, 2, 2), 10, "off", 3), (4, 3, (1, 2, 1, 2), 1, "type1", 2),
         (4, 4, (1, 2, 2, 2), 0, "v", 2), (5, 4, (1, 2, 2, 2), 10, "skew", 2), (7, 7, (1, 2, 2, 2), 10, "ga", 1)]


@pytest.mark.parametrize("D,L,law,type_,kind,nvec", CASES)
def test_hterm(evr, oracle_mod, D, L, law, type_, kind, nvec):
    rng = np.random.RandomState(D * 100 + L)
    s = oracle_mod.SG4(D, L, L, *law)
    b = evr.Basis.sg4(D, L, L, *law)
    G0 = np.diag(rng.uniform(1.0, 3.0, D))
    if kind != "g0":
        G0 = G0 + 0.1 * rng.uniform(-1.0, 1.0, (D, D))
    Ga = F1 = None
    if kind in ("ga", "skew"):
        Ga = rng.uniform(-0.1, 0.1, (D, D, D))
        if kind == "ga":
            Ga = 0.5 * (Ga + Ga.transpose(1, 0, 2))  # G_ij(q) = G_ji(q)
        Ga = Ga.ravel(order="F")
    if type_ == 1:
        F1 = rng.uniform(-0.1, 0.1, D)
    q = s.grid()
    V = 0.5 * (q ** 2).sum(axis=1) + 0.1 * q[:, 0] * q[:, -1] ** 2
    X = np.asfortranarray(rng.randn(b.nb_packed, nvec))
    if type_ == 10:
        op, kw = oracle_mod.Op(10, V=V, G0=G0, Ga=Ga), dict(G0=G0, Ga=Ga)
    elif type_ == 1:
        op, kw = oracle_mod.Op(1, V=V, F2=G0, F1=F1), dict(F2=G0, F1=F1)
    else:
        op, kw = oracle_mod.Op(0, V=V), {}
    ref = s.oppsi(op, X)
    plan = evr.Plan(b, type=type_, V=V, max_nvec=nvec, **kw)
    e = np.abs(plan.TabOpPsi(X) - ref).max() / np.abs(ref).max()
    print("D=%d L=%d law %s type %d %s, %d vectors: %.2e" % (D, L, law, type_, kind, nvec, e))
    assert e < TOL64


@pytest.mark.parametrize("D,L,law,ncol", [(1, 3, (1, 2, 2, 2), 1), (2, 9, (1, 2, 2, 2), 2), (4, 4, (1, 2, 1, 2), 2),
                                          (4, 3, (1, 1, 2, 1), 2), (3, 3, (2, 2, 3, 2), 3), (6, 5, (1, 2, 2, 2), 5),
                                          (7, 7, (1, 2, 2, 2), 1), (9, 4, (1, 2, 2, 2), 2), (12, 3, (1, 2, 2, 2), 1),
                                          (12, 2, (1, 2, 1, 2), 3)])
def test_transforms(evr, oracle_mod, D, L, law, ncol):
    """Basis -> grid and the weighted grid -> basis in register blocks: few and
    many one-function modes, their points below and above the low part of 128,
    terms whose reduced grid stays with the term kernels (seven modes)."""
    s = oracle_mod.SG4(D, L, L, *law)
    b = evr.Basis.sg4(D, L, L, *law)
    # a q-linear G: the H|psi> tables of such a plan are rotated, these are not
    plan = evr.Plan(b, type=10, G0=np.eye(D), Ga=np.full(D ** 3, 0.01), max_nvec=ncol)
    rng = np.random.RandomState(D * 10 + L)
    X = np.asfortranarray(rng.randn(b.nb_packed, ncol))
    G = plan.BasisRep_TO_GridRep_n(X)
    for c in range(ncol):
        ref = s.b2g(X[:, c])
        assert np.abs(G[:, c] - ref).max() / np.abs(ref).max() < TOL64
    Gr = np.asfortranarray(rng.randn(b.sum_nq, ncol))
    Y = plan.GridRep_TO_BasisRep_n(Gr)
    for c in range(ncol):
        ref = s.g2b(Gr[:, c])
        assert np.abs(Y[:, c] - ref).max() / np.abs(ref).max() < TOL64


def q_linear(D, rng, symmetric):
    G0 = np.diag(rng.uniform(1.0, 3.0, D))
    Ga = rng.uniform(-0.1, 0.1, (D, D, D))
    if symmetric:  # in all three indices, as the hermitian form needs
        Ga = sum(Ga.transpose(p) for p in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))) / 6.0
        for i, j, k in np.ndindex(D, D, D):
            Ga[i, j, k] = Ga[tuple(sorted((i, j, k)))]
    else:
        Ga = 0.5 * (Ga + Ga.transpose(1, 0, 2))
    return G0, Ga.ravel(order="F")


@pytest.mark.parametrize("D,L,law,nvec", [
    (1, 11, (1, 1, 2, 1), 3),                            # one mode, one group of any shape (12 functions)
    (2, 8, (1, 2, 2, 2), 5),                             # one group of any shape beside a table shape, and none
    (3, 2, (2, 2, 3, 2), 8), (3, 2, (2, 2, 3, 2), 33),   # three: the classes in one launch, and in several
    (4, 3, (2, 2, 3, 2), 1), (4, 3, (2, 2, 3, 2), 17),   # four
    (2, 1, (30, 1, 31, 1), 2)])                          # 30 and 31 functions
def test_any_shape(evr, oracle_mod, D, L, law, nvec):
    """Rotations of groups outside the table of shapes, in odd and even number,
    and launches that several classes share."""
    rng = np.random.RandomState(D + L + nvec)
    s = oracle_mod.SG4(D, L, L, *law)
    b = evr.Basis.sg4(D, L, L, *law)
    G0, Ga = q_linear(D, rng, False)
    q = s.grid()
    V = 0.5 * (q ** 2).sum(axis=1) + 0.1 * q[:, 0] * q[:, -1] ** 2
    X = np.asfortranarray(rng.randn(b.nb_packed, nvec))
    ref = s.oppsi(oracle_mod.Op(10, V=V, G0=G0, Ga=Ga), X)
    e = np.abs(evr.Plan(b, type=10, V=V, G0=G0, Ga=Ga, max_nvec=nvec).TabOpPsi(X) - ref).max() / np.abs(ref).max()
    print("D=%d L=%d law %s, %d vectors: %.2e" % (D, L, law, nvec, e))
    assert e < TOL64


@pytest.mark.parametrize("D,L,law,nvec", [(3, 4, (1, 2, 2, 2), 3), (5, 3, (1, 2, 1, 2), 8), (4, 2, (2, 1, 3, 1), 2)])
def test_hermitian(evr, oracle_mod, D, L, law, nvec):
    """The symmetric form of a q-linear G, (H + H^T) / 2 of the oracle's H."""
    rng = np.random.RandomState(7 * D + L)
    s = oracle_mod.SG4(D, L, L, *law)
    b = evr.Basis.sg4(D, L, L, *law)
    G0, Ga = q_linear(D, rng, True)
    q = s.grid()
    V = 0.5 * (q ** 2).sum(axis=1) + 0.1 * q[:, 0] * q[:, -1] ** 2
    X = np.asfortranarray(rng.randn(b.nb_packed, nvec))
    M = s.oppsi(oracle_mod.Op(10, V=V, G0=G0, Ga=Ga), np.asfortranarray(np.eye(b.nb_packed)))
    ref = 0.5 * (M @ X + M.T @ X)
    plan = evr.Plan(b, type=10, V=V, G0=G0, Ga=Ga, max_nvec=nvec, hermitian=True)
    e = np.abs(plan.TabOpPsi(X) - ref).max() / np.abs(ref).max()
    print("D=%d L=%d law %s, %d vectors: %.2e" % (D, L, law, nvec, e))
    assert e < TOL64


def test_brackets_in_passes(evr, oracle_mod):
    """Terms whose brackets of all modes do not fit the LDS beside x and y: the
    kinetic part takes them a few modes at a time."""
    D, nvec = 4, 2
    s = oracle_mod.SG4(D, 1, 1, 8, 1, 9, 1)
    b = evr.Basis.sg4(D, 1, 1, 8, 1, 9, 1)
    assert 8 * (2 + D) * 8 ** 4 > 160 * 1024 > 8 * (3 * 9 * 8 ** 3 + 2000)
    rng = np.random.RandomState(5)
    G0, Ga = q_linear(D, rng, False)
    q = s.grid()
    V = 0.5 * (q ** 2).sum(axis=1) + 0.1 * q[:, 0] * q[:, -1] ** 2
    X = np.asfortranarray(rng.randn(b.nb_packed, nvec))
    ref = s.oppsi(oracle_mod.Op(10, V=V, G0=G0, Ga=Ga), X)
    plan = evr.Plan(b, type=10, V=V, G0=G0, Ga=Ga, max_nvec=nvec)
    plan.set_profiling(True)
    Y = plan.TabOpPsi(X)
    assert [n for n, _, _, k in plan.kernel_stats() if k] == ["k_hterm"]
    e = np.abs(Y - ref).max() / np.abs(ref).max()
    print("%.2e" % e)
    assert e < TOL64


@pytest.mark.parametrize("D,L,law,ncol", [
    (10, 2, (1, 1, 1, 1), 5),     # grids of up to 4 points: a wave per term
    (4, 4, (1, 2, 2, 2), 3),      # up to 256 points: four waves
    (4, 4, (1, 2, 2, 2), 40)])    # the same in many workgroups: one wave
def test_transform_workgroups(evr, oracle_mod, D, L, law, ncol):
    """Transforms in workgroups of one wave and of four."""
    s = oracle_mod.SG4(D, L, L, *law)
    b = evr.Basis.sg4(D, L, L, *law)
    plan = evr.Plan(b, type=0, max_nvec=ncol)
    rng = np.random.RandomState(D + ncol)
    X = np.asfortranarray(rng.randn(b.nb_packed, ncol))
    Gr = np.asfortranarray(rng.randn(b.sum_nq, ncol))
    G, Y = plan.BasisRep_TO_GridRep_n(X), plan.GridRep_TO_BasisRep_n(Gr)
    for c in range(ncol):
        ref = s.b2g(X[:, c])
        assert np.abs(G[:, c] - ref).max() / np.abs(ref).max() < TOL64
        ref = s.g2b(Gr[:, c])
        assert np.abs(Y[:, c] - ref).max() / np.abs(ref).max() < TOL64


@pytest.mark.parametrize("D,L,law,nvec,kernel", [
    (6, 7, (1, 2, 2, 2), 1, "k_hterm"),       # 110 us, assembled 169 us
    (6, 7, (1, 2, 2, 2), 32, "k_apply_asm"),  # 523 us, assembled 226 us
    (4, 1, (8, 1, 9, 1), 2, "k_apply_asm"),   # five terms, the chain of one: 449 us, assembled 234 us
    (6, 4, (2, 2, 3, 2), 4, "k_apply_asm")])  # shapes outside the table: 192 us, assembled 125 us
def test_auto_path(evr, D, L, law, nvec, kernel):
    """The automatic choice takes the path that is the faster one by far."""
    b = evr.Basis.sg4(D, L, L, *law)
    plan = evr.Plan(b, type=10, V=0.5 * (b.grid() ** 2).sum(1), G0=np.eye(D), Ga=np.full(D ** 3, 0.01),
                    max_nvec=nvec, hermitian=True)
    plan.assemble(evr.ASM_FP64)
    X = evr.hamiltonian.test_vectors(b.nb_packed, nvec, 3)
    ref = plan.TabOpPsi(X, evr.MATRIX_FREE)
    plan.set_profiling(True)
    Y = plan.TabOpPsi(X, evr.AUTO_PATH)
    assert [n for n, _, _, k in plan.kernel_stats() if k] == [kernel]
    assert np.abs(Y - ref).max() / np.abs(ref).max() < TOL64
