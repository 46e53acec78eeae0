"""The block-form MPO-term sum at the edges of its work splits, against the CPU oracle: tiles of
s x s elements with s*s around 32 (one wave), 64 (two waves) and 128 (a workgroup's range), single
elements, odd sizes (an element pair past the tile's end) and coefficient tables longer than one
staging pass.  FP64 to 1e-12 of the largest element (sums of a few thousand products, 2^-53 each),
FP32 to 1e-5 (the mixed-precision bound of the other parity tests).  The same term by term, at the edges
of its lane groups and of the shares of a line's terms (lines of 1 to several hundred terms)."""
import numpy as np
import pytest

from qcmaquis_amd import abi
from qcmaquis_amd.engine import DeviceBoundary, DeviceMPO, HpsiPlan
from qcmaquis_amd.synthetic import TWOU1_SITE, Chain, fuse_index
from tests.chains import oracle_left, oracle_right, rel_err

pytestmark = pytest.mark.gpu


def problem(oracle_lib, s, D):
    ch = Chain(np.random.default_rng(100 + s), abi.MQ_SYM_TWOU1, 4, (4, 4), s, D,
               phys=fuse_index(TWOU1_SITE, TWOU1_SITE), density=0.5, min_m=s)
    k = 2
    L = oracle_left(oracle_lib, ch, k)[k]
    R = oracle_right(oracle_lib, ch, k + 1)[k + 1]
    lay = ch.layouts[k]
    return ch.sym, ch.mpos[k], L, R, lay, np.random.default_rng(s).normal(size=lay.n)


def make_plan(ctx, mpo, L, R, lay, small_max):
    ctx.set_option(abi.MQ_OPT_SMALL_TILE_MAX, small_max)
    try:
        return HpsiPlan(ctx, DeviceMPO(ctx, mpo), DeviceBoundary.upload(ctx, L), DeviceBoundary.upload(ctx, R), lay)
    finally:
        ctx.set_option(abi.MQ_OPT_SMALL_TILE_MAX, abi.MQ_SMALL_TILE_AUTO)


def run(oracle_lib, ctx, s, D, small_max):
    sym, mpo, L, R, lay, psi = problem(oracle_lib, s, D)
    ref = oracle_lib.hpsi(sym, mpo, L, R, lay, psi)
    plan = make_plan(ctx, mpo, L, R, lay, small_max)
    st = plan.stats()
    err = rel_err(plan.apply(psi), ref)
    err32 = rel_err(plan.apply(psi, abi.MQ_PREC_FP32), ref)
    print(f"tiles {s}x{s}: {st['n_sblocks']} blocks, {st['small_lines']} small lines, max union {st['max_union_tiles']}, "
          f"FP64 {err:.1e}, FP32 {err32:.1e}", flush=True)
    return st, err, err32


@pytest.mark.parametrize("s,D", [(s, 24) for s in (1, 2, 5, 6, 8, 9, 11, 12, 17)] + [(s, 64) for s in (1, 5, 6, 8, 12)])
def test_block_sum_tile_sizes(oracle_lib, ctx2u1, s, D):
    st, err, err32 = run(oracle_lib, ctx2u1, s, D, 0)  # every tile in blocks
    assert st["small_lines"] == 0 and st["n_sblocks"] > 0
    # 64 k-steps of four tiles: shared out in tiles of up to 64 elements, more than one staging pass in larger ones
    assert D < 64 or st["max_union_tiles"] >= 4 * 64 + (s > 8)
    assert err < 1e-12 and err32 < 1e-5


@pytest.mark.parametrize("s,D", [(1, 24), (1, 64), (2, 64), (3, 24), (5, 24), (8, 64), (9, 24), (11, 64), (16, 64)])
def test_small_line_groups(oracle_lib, ctx2u1, s, D):
    st, err, err32 = run(oracle_lib, ctx2u1, s, D, 256)  # every tile term by term
    assert st["n_sblocks"] == 0 and st["small_lines"] > 0
    assert err < 1e-12 and err32 < 1e-5


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("s,D", [(1, 24), (5, 24), (8, 24), (1, 64), (6, 64)])
def test_non_finite_elements(oracle_lib, ctx2u1, s, D, value):
    """an infinite or undefined psi element reaches the same elements of H*psi whether tiles of at most 64
    elements are summed in blocks or term by term, i.e. only those whose lines read it; the others agree to
    1e-12 (FP64) and 1e-5 (FP32) of the largest of them"""
    sym, mpo, L, R, lay, psi = problem(oracle_lib, s, D)
    plans = [make_plan(ctx2u1, mpo, L, R, lay, m) for m in (256, 0)]
    few = 0
    for at in (0, lay.n // 2, lay.n - 1):
        x = psi.copy()
        x[at] = value
        for prec, tol in ((abi.MQ_PREC_FP64, 1e-12), (abi.MQ_PREC_FP32, 1e-5)):
            terms, blocks = (p.apply(x, prec) for p in plans)
            ok = np.isfinite(terms)
            print(f"tiles {s}x{s}, psi[{at}] = {value}: {ok.sum()} of {lay.n} finite, in blocks {np.isfinite(blocks).sum()}",
                  flush=True)
            assert np.array_equal(ok, np.isfinite(blocks))
            assert not ok.any() or rel_err(blocks[ok], terms[ok]) < tol
            few += 0 < ok.sum() < lay.n
    assert few > 0
