"""The grouped GEMMs at the edges of their work items, against the CPU oracle: sectors of s states
around the 16-row steps of a wave, the tile heights 32, 64, 96 and 128, the 128 columns of an item
and, as reduction lengths, the K slices of 16.  Left growth takes A transposed, right growth B (in products
that may be split along K; H*psi has B transposed in stacked ones).  FP64 to 1e-12 of the largest
element (sums of a few thousand products, 2^-53 each), FP32 to 1e-5 and split BF16 to 5e-4 (the bounds
of the other parity tests)."""
import numpy as np
import pytest

from qcmaquis_amd import abi
from qcmaquis_amd.engine import DeviceBoundary, DeviceMPO, DeviceMPS, HpsiPlan, lstep, rstep
from qcmaquis_amd.synthetic import Chain
from tests.chains import oracle_left, oracle_right, rel_err

pytestmark = pytest.mark.gpu


# (12, 96), (17, 64) and (33, 48): reductions of a few thousand, split into more than eight ranges
@pytest.mark.parametrize("s,D", [(s, 6) for s in (1, 3, 15, 16, 17, 31, 33, 64, 65, 97, 127, 128, 129, 140)] +
                         [(12, 96), (17, 64), (33, 48)])
def test_gemm_tile_edges(oracle_lib, ctx2u1, s, D):
    ch = Chain(np.random.default_rng(200 + s), abi.MQ_SYM_TWOU1, 4, (2, 2), s, D, min_m=s)
    k = 2
    L = oracle_left(oracle_lib, ch, k + 1)
    R = oracle_right(oracle_lib, ch, k)
    lay = ch.layouts[k]
    psi = np.random.default_rng(s).normal(size=lay.n)
    ref = oracle_lib.hpsi(ch.sym, ch.mpos[k], L[k], R[k + 1], lay, psi)
    dl, dr, mpo = DeviceBoundary.upload(ctx2u1, L[k]), DeviceBoundary.upload(ctx2u1, R[k + 1]), DeviceMPO(ctx2u1, ch.mpos[k])
    plan = HpsiPlan(ctx2u1, mpo, dl, dr, lay)
    err = rel_err(plan.apply(psi), ref)
    err32 = rel_err(plan.apply(psi, abi.MQ_PREC_FP32), ref)
    err16 = rel_err(plan.apply(psi, abi.MQ_PREC_BF16X3), ref)
    site = DeviceMPS(ctx2u1, lay, ch.data[k])
    grown = lstep(ctx2u1, mpo, dl, site, site, True).download()
    err_l = rel_err(grown.data, L[k + 1].data)
    err_r = rel_err(rstep(ctx2u1, mpo, dr, site, site, True).download().data, R[k].data)
    print(f"sectors of {s}: FP64 {err:.1e}, FP32 {err32:.1e}, split BF16 {err16:.1e}, growth {err_l:.1e} and {err_r:.1e}",
          flush=True)
    assert err < 1e-12 and err32 < 1e-5 and err16 < 5e-4 and err_l < 1e-12 and err_r < 1e-12
