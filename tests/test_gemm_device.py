"""The device form of the grouped GEMM stages against the plan's own problems, on the CPU."""
import ctypes as C
import math
import os
import subprocess

import pytest

from qcmaquis_amd import abi
from qcmaquis_amd.synthetic import TWOU1_SITE, fuse_index
from tests import emu
from tests.chains import make_chain, oracle_left, oracle_right

LIB = os.path.join(emu.HERE, "libgemmdevice.so")


@pytest.fixture(scope="module")
def lib():
    srcs = [os.path.join(emu.HERE, "gemm_device.cpp")] + [os.path.join(emu.CSRC, f) for f in
                                                          ("plans.cpp", "coupling.cpp", "descriptors.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fopenmp", "-I", os.path.join(emu.ROOT, "include"),
                    "-I", emu.CSRC, "-o", LIB] + srcs, check=True)
    lib = C.CDLL(LIB)
    idx = C.POINTER(abi.IndexDesc)
    lib.fold_check.restype = C.c_long
    lib.fold_check.argtypes = [C.c_int, C.POINTER(abi.MPODesc), C.POINTER(abi.BIndexDesc), C.POINTER(abi.BIndexDesc), idx,
                               idx, idx]
    ints = C.POINTER(C.c_int)
    lib.items_check.restype = C.c_long
    lib.items_check.argtypes = [C.c_int, ints, ints, ints, C.c_int, C.c_int]
    lib.candidate_policies.restype = C.c_long
    lib.candidate_policies.argtypes = [C.c_int, ints, ints, ints, C.c_int, C.c_int]
    lib.stage_key.restype = C.c_uint64
    lib.stage_key.argtypes = [C.c_int, ints, ints, ints, C.c_int, C.POINTER(C.c_long)]
    lib.fold_columns.argtypes = [C.c_int, C.c_int, C.POINTER(C.c_long), C.POINTER(C.c_long)]
    return lib


CHAINS = [
    (abi.MQ_SYM_TWOU1, 1, dict(n_sites=5, total=(3, 2), max_m=1, D=6)),
    (abi.MQ_SYM_TWOU1, 2, dict(n_sites=5, total=(3, 2), max_m=9, D=9)),
    (abi.MQ_SYM_TWOU1, 3, dict(n_sites=4, total=(4, 4), max_m=7, D=12, phys=fuse_index(TWOU1_SITE, TWOU1_SITE))),
    (abi.MQ_SYM_SU2U1, 4, dict(n_sites=5, total=(4, 0), max_m=6, D=9)),
]


def test_folded_batches(oracle_lib, lib):
    folded = 0
    for sym, seed, kw in CHAINS:
        ch = make_chain(seed, sym=sym, **kw)
        n = len(ch.mpos)
        L, R = oracle_left(oracle_lib, ch, n - 1), oracle_right(oracle_lib, ch, 1)
        for k in range(n):
            lay = ch.layouts[k]
            d = [ch.mpos[k].desc(), L[k].desc(), R[k + 1].desc(), lay.left.desc(), lay.phys.desc(), lay.right.desc()]
            f = lib.fold_check(sym, *[C.byref(x) for x in d])
            assert f >= 0, (sym, seed, k)
            folded += f
    assert folded > 0


@pytest.mark.parametrize("policy", range(7))
def test_work_items(lib, policy):
    """tiles, K splits and partials over sizes around the tile heights, widths and K steps"""
    m = [1, 15, 32, 33, 64, 96, 97, 128, 129, 200, 257, 300]
    n = [1, 16, 127, 128, 129, 300, 5, 40, 260, 64, 33, 130]
    k = [1, 17, 256, 1000, 513, 3, 16, 700, 2049, 128, 4000, 31]
    arr = [(C.c_int * len(v))(*v) for v in (m, n, k)]
    assert lib.items_check(len(m), *arr, 2, policy) > 0


@pytest.mark.parametrize("flags,batch", [(4, 1), (6, 5), (0, 1)])  # GEMM_ROWMAP, with GEMM_TRANS_B, plain
def test_autotuner_candidates(lib, flags, batch):
    """a stage whose schedules are all alike (stacked problems, which K is not split for, and reductions
    too short to be split) has the default rule only; the others have every schedule once"""
    arr = lambda *v: (C.c_int * len(v))(*v)
    long_k = (arr(64, 130, 97), arr(300, 128, 5), arr(9000, 4000, 2049))
    short_k = (arr(64, 130), arr(300, 128), arr(100, 16))
    assert lib.candidate_policies(2, *short_k, batch, flags) == 1
    bits = lib.candidate_policies(3, *long_k, batch, flags)
    assert bits == 1 if flags & 4 else bits & 1 and bin(bits).count("1") > 2


@pytest.mark.parametrize("m,n,k", [((128,), (128,), (700,)), ((129,), (64,), (300,)), ((200, 300), (1000, 65), (50, 4000)),
                                   ((33, 1, 97), (5, 4000, 257), (100, 9, 3))])
def test_stage_key_counts_tiles(lib, m, n, k):
    """the tile count in a stage's key (log2, bits 1 to 6) is the one of the schedule"""
    arr, tiles = [(C.c_int * len(v))(*v) for v in (m, n, k)], C.c_long()
    key = lib.stage_key(len(m), *arr, 8, C.byref(tiles))
    assert tiles.value > 0 and (key - 1) >> 1 & 63 == math.floor(math.log2(tiles.value) + 0.5)


@pytest.mark.parametrize("n,batch,fold", [(5, 7, True), (16777215, 128, False), (1073741821, 2, False),
                                          (67108863, 32, False), (65535, 32766, True)])
def test_folded_columns_fit(lib, n, batch, fold):
    """blocks are folded only while the rounded-up column count is a 32-bit number"""
    cols, tiles = C.c_long(), C.c_long()
    lib.fold_columns(n, batch, C.byref(cols), C.byref(tiles))
    assert cols.value == (n * batch if fold else n) and tiles.value == -(-cols.value // 128)
