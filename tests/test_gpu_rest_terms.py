"""Plans in which some terms run in register blocks and others stay with the
term kernels: FP64 H|psi> (terms of nine active modes beside terms of eight) and
the FP64 transforms (a reduced grid of 5^6 points beyond a workgroup's LDS),
under the static classes, with every bucket of terms moved to larger classes,
and after a tuning run, against the oracle.  The kernel that a remaining term
runs in is always the one its class names."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL64 = 1e-12  # the parity bar of every FP64 H|psi> test
TOL32 = 2e-5   # and of FP32 ones

CLASSES = ["k_term<256,1,4>", "k_term<512,1,4>", "k_term<512,2,4>", "k_term<512,2,2>", "k_term<512,4,2>",
           "k_term<512,4,1>", "k_term<1024,4,1>", "k_term<1024,8,1>"]
MAX_NBT = [64, 128, 256, 512, 1024, 2048, 4096, 8192]
PICKS = [[min(b + 1, 7) for b in range(8)], [min(b + 2, 7) for b in range(8)], list(range(8))]


def operator(D, seed):
    rng = np.random.RandomState(seed)
    G0 = np.diag(rng.uniform(1.0, 3.0, D)) + 0.1 * np.ones((D, D))
    Ga = rng.uniform(-0.1, 0.1, (D, D, D))
    return G0, (0.5 * (Ga + Ga.transpose(1, 0, 2))).ravel(order="F")


def setup(evr, oracle_mod, D, L, law, nvec):
    s = oracle_mod.SG4(D, L, L, *law)
    b = evr.Basis.sg4_modes(D, L, *law)
    G0, Ga = operator(D, D)
    q = s.grid()
    V = 0.5 * (q ** 2).sum(axis=1) + 0.1 * q[:, 0] * q[:, -1] ** 2
    plan = evr.Plan(b, type=10, V=V, G0=G0, Ga=Ga, max_nvec=nvec)
    return s, b, plan, oracle_mod.Op(10, V=V, G0=G0, Ga=Ga)


def set_classes(evr, plan, pick):
    evr._lib.check(evr._lib.load().evr_plan_set_classes(plan.h, (ctypes.c_int * 8)(*pick)))


def launched(plan, call):
    """Names of the profiled kernels that the call launched."""
    plan.set_profiling(True)
    call()
    names = {n for n, _, _, launches in plan.kernel_stats() if launches}
    plan.set_profiling(False)
    return names


def relerr(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def test_hpsi_follows_the_classes(evr, oracle_mod):
    nvec = 5
    # mode 9 has one function at level 0 (eight active modes) and two at level
    # 1 (nine: 512 functions with all the others at their two)
    law = ([2] * 8 + [1], [1] * 9, [3] * 8 + [2], [1] * 9)
    s, b, plan, op = setup(evr, oracle_mod, 9, 1, law, nvec)
    X = np.asfortranarray(np.random.RandomState(3).randn(b.nb_packed, nvec))
    ref = s.oppsi(op, X)

    def check(what):
        e = relerr(plan.TabOpPsi(X), ref)
        e32 = relerr(plan.TabOpPsi(X, flags=evr.FP32), ref)
        print("%s: %.2e, FP32 %.2e" % (what, e, e32))
        assert e < TOL64 and e32 < TOL32

    check("static")
    home = next(c for c in range(8) if MAX_NBT[c] >= 512)
    assert launched(plan, lambda: plan.TabOpPsi(X)) == {"k_hterm", CLASSES[home]}
    for pick in PICKS:
        set_classes(evr, plan, pick)
        assert launched(plan, lambda: plan.TabOpPsi(X)) == {"k_hterm", CLASSES[pick[home]]}
        check("classes %s" % pick)
    for flags in (evr.FP32, evr.FP64):
        plan.autotune(nvec, flags, reps=1)
        check("tuned")


def test_transforms_follow_the_classes(evr, oracle_mod):
    ncol = 2
    s, b, plan, _ = setup(evr, oracle_mod, 6, 6, ([1] * 6, [1] * 6, [3] * 6, [2] * 6), ncol)
    rng = np.random.RandomState(4)
    X = np.asfortranarray(rng.randn(b.nb_packed, ncol))
    Gr = np.asfortranarray(rng.randn(b.sum_nq, ncol))
    rb = [s.b2g(X[:, c]) for c in range(ncol)]
    rg = [s.g2b(Gr[:, c]) for c in range(ncol)]

    def check(what):
        G = plan.BasisRep_TO_GridRep_n(X)
        Y = plan.GridRep_TO_BasisRep_n(Gr)
        e = max(relerr(G[:, c], rb[c]) for c in range(ncol))
        eg = max(relerr(Y[:, c], rg[c]) for c in range(ncol))
        print("%s: %.2e, back %.2e" % (what, e, eg))
        assert e < TOL64 and eg < TOL64

    check("static")
    for pick in PICKS:
        set_classes(evr, plan, pick)
        # the 5^6 term has 64 functions, the first class's most
        assert launched(plan, lambda: plan.BasisRep_TO_GridRep_n(X)) == {"k_b2g", CLASSES[pick[0]]}
        assert launched(plan, lambda: plan.GridRep_TO_BasisRep_n(Gr)) == {"k_g2b", CLASSES[pick[0]]}
        check("classes %s" % pick)
    plan.autotune(ncol, evr.FP32, reps=1)
    check("tuned")


def test_class_below_a_bucket_is_refused(evr, oracle_mod):
    _, _, plan, _ = setup(evr, oracle_mod, 3, 2, ([1] * 3, [2] * 3, [2] * 3, [2] * 3), 1)
    with pytest.raises(RuntimeError, match="class"):
        set_classes(evr, plan, [0] * 8)
