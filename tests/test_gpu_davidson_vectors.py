"""The Jacobi-Davidson's vector kernels at the edges of their launches (16 vectors in one linear
combination or product launch, the coefficients of 32 batch instances): the energy after a fixed number
of iterations against the same iteration in numpy on the oracle's dense operator, and a batch of 35
against it too.  Both sides run one recursion in FP64; with the operator's elements off by 1e-15 the
numpy side's energies move by at most 2e-12 (20 iterations), so 1e-10 bounds them."""
import numpy as np
import pytest

from qcmaquis_amd import abi
from qcmaquis_amd.engine import DeviceBoundary, DeviceMPO, HpsiPlan, HpsiPlanBatch
from tests.chains import make_chain, oracle_left, oracle_right

pytestmark = pytest.mark.gpu


def jd(H, x, iters):
    """energy after `iters` iterations: Gram-Schmidt, Ritz pair, residual, correction"""
    V, W, t = [], [], x.copy()
    for _ in range(iters):
        for _ in range(2):
            for v in V:
                t = t - (v @ t) * v
        V.append(t / np.linalg.norm(t))
        W.append(H @ V[-1])
        M = np.array([[v @ w for w in W] for v in V])  # its upper half counts (H of a random chain is not symmetric)
        e, s = np.linalg.eigh(np.triu(M) + np.triu(M, 1).T)
        u, uA = np.array(V).T @ s[:, 0], np.array(W).T @ s[:, 0]
        r = uA - e[0] * u
        t = -r + (r @ u) / (u @ u) * u
    return e[0]


@pytest.fixture(scope="module")
def site(oracle_lib, ctx2u1):
    ch = make_chain(11, n_sites=4, total=(2, 2), max_m=9, D=6)
    k = 2
    L, R = oracle_left(oracle_lib, ch, k)[k], oracle_right(oracle_lib, ch, k + 1)[k + 1]
    lay = ch.layouts[k]
    H = np.array([oracle_lib.hpsi(ch.sym, ch.mpos[k], L, R, lay, e) for e in np.eye(lay.n)]).T
    item = (DeviceMPO(ctx2u1, ch.mpos[k]), DeviceBoundary.upload(ctx2u1, L), DeviceBoundary.upload(ctx2u1, R), lay)
    return H, item


@pytest.mark.parametrize("iters", [1, 2, 3, 15, 16, 17, 20])
def test_iterations(ctx2u1, site, iters):
    H, item = site
    n = item[3].n
    assert n > 40
    x = np.random.default_rng(iters).normal(size=n)
    e, v, st = HpsiPlan(ctx2u1, *item).davidson(x, tol=1e-300, max_iter=iters)
    ref = jd(H, x, iters)
    print(f"{iters} iterations, n = {n}: {e:.12f} {ref:.12f}", flush=True)
    assert st["iterations"] == iters
    assert abs(e - ref) <= 1e-10 * abs(ref)


def test_batch_of_35(ctx2u1, site):
    H, item = site
    rng = np.random.default_rng(5)
    xs = [rng.normal(size=item[3].n) for _ in range(35)]
    batch = HpsiPlanBatch(ctx2u1, [item] * 35)
    for iters in (1, 4, 17):
        e, vs, its, _ = batch.davidson(xs, tol=1e-300, max_iter=iters)
        ref = [jd(H, x, iters) for x in xs]
        err = max(abs(a - b) / abs(b) for a, b in zip(e, ref))
        print(f"35 instances, {iters} iterations: {err:.1e}", flush=True)
        assert list(its) == [iters] * 35 and err <= 1e-10
