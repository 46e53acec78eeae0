"""The grouped GEMMs at the edges of their work items, against the CPU oracle: sectors of s states
around the 16-row steps of a wave, the tile heights 32, 64, 96 and 128, the 128 columns of an item
and, as reduction lengths, the K slices of 16.  A growth step takes the transposed orientations.
FP64 to 1e-12 of the largest element (sums of a few thousand products, 2^-53 each), FP32 to 1e-5
(the mixed-precision bound of the other parity tests)."""
import numpy as np
import pytest

from qcmaquis_amd import abi
from qcmaquis_amd.engine import DeviceBoundary, DeviceMPO, DeviceMPS, HpsiPlan, lstep
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
    R = oracle_right(oracle_lib, ch, k + 1)[k + 1]
    lay = ch.layouts[k]
    psi = np.random.default_rng(s).normal(size=lay.n)
    ref = oracle_lib.hpsi(ch.sym, ch.mpos[k], L[k], R, lay, psi)
    dl, mpo = DeviceBoundary.upload(ctx2u1, L[k]), DeviceMPO(ctx2u1, ch.mpos[k])
    plan = HpsiPlan(ctx2u1, mpo, dl, DeviceBoundary.upload(ctx2u1, R), lay)
    err = rel_err(plan.apply(psi), ref)
    err32 = rel_err(plan.apply(psi, abi.MQ_PREC_FP32), ref)
    site = DeviceMPS(ctx2u1, lay, ch.data[k])
    grown = lstep(ctx2u1, mpo, dl, site, site, True).download()
    err_l = rel_err(grown.data, L[k + 1].data)
    print(f"sectors of {s}: FP64 {err:.1e}, FP32 {err32:.1e}, growth {err_l:.1e}", flush=True)
    assert err < 1e-12 and err32 < 1e-5 and err_l < 1e-12
