"""H|psi> of direct-product terms in three passes (two groups of modes) against
the oracle: two to four modes, extents below, at and above the 16 outputs and 4
inputs of a matrix tile, up to 64 points, one to many vectors, with and without
cross terms in the kinetic part, and without a potential."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL64 = 1e-12  # the parity bar of every FP64 H|psi> test

CASES = [((16, 16), (16, 17), "ga", 1), ((40, 17), (41, 18), "g0", 3), ((31, 63), (33, 64), "ga", 5),
         ((7, 9, 5), (8, 9, 6), "off", 2), ((12, 12, 12), (14, 14, 14), "g0", 1), ((17, 3, 33), (18, 4, 34), "ga", 7),
         ((40, 33, 7), (41, 35, 9), "type1", 3), ((8, 40, 40), (8, 41, 41), "ga", 1), ((13, 11, 9), (14, 13, 10), "v", 2),
         ((5, 4, 6, 7), (6, 4, 8, 8), "ga", 3), ((4, 16, 5, 17), (5, 17, 6, 18), "type1", 2),
         ((6, 5, 20, 9), (7, 6, 21, 10), "g0", 9), ((9, 3, 33, 4), (9, 4, 34, 5), "off", 33),
         ((5, 4, 3, 40), (5, 5, 4, 42), "diag1", 4), ((7, 7, 7), (8, 8, 8), "nov", 2)]


@pytest.mark.parametrize("nb,nq,kind,nvec", CASES)
def test_three_passes(evr, oracle_mod, nb, nq, kind, nvec):
    D = len(nb)
    rng = np.random.RandomState(sum(nb) + nvec)
    d = oracle_mod.DP(list(nb), list(nq))
    b = evr.Basis.dp(list(nb), list(nq))
    q = d.grid()
    G0 = np.diag(rng.uniform(1.0, 3.0, D))
    if kind not in ("g0", "diag1", "nov"):
        G0 = G0 + 0.1 * rng.uniform(-1.0, 1.0, (D, D))
    V = 0.5 * (q ** 2).sum(axis=1) + 0.1 * q[:, 0] * q[:, -1] ** 2
    X = np.asfortranarray(rng.randn(b.nb_packed, nvec))
    if kind in ("type1", "diag1"):
        F1 = rng.uniform(-0.1, 0.1, D)
        op, kw, type_ = oracle_mod.Op(1, V=V, F2=G0, F1=F1), dict(F2=G0, F1=F1), 1
    elif kind == "v":
        op, kw, type_ = oracle_mod.Op(0, V=V), {}, 0
    else:
        Ga = rng.uniform(-0.1, 0.1, (D, D, D)).ravel(order="F") if kind in ("ga", "nov") else None
        op = oracle_mod.Op(10, V=0.0 * V if kind == "nov" else V, G0=G0, Ga=Ga)
        kw, type_ = dict(G0=G0, Ga=Ga), 10
    ref = d.oppsi(op, X)
    plan = evr.Plan(b, type=type_, V=None if kind == "nov" else V, max_nvec=nvec, **kw)
    e = np.abs(plan.TabOpPsi(X) - ref).max() / np.abs(ref).max()
    e1 = np.abs(plan.TabOpPsi(X[:, :1]) - ref[:, :1]).max() / np.abs(ref).max()
    print("%s on %s, %s, %d vectors: %.2e, one %.2e" % (nb, nq, kind, nvec, e, e1))
    assert e < TOL64 and e1 < TOL64
