"""Timed cases of the contraction path: H*psi, Davidson, boundary growth and integral gradients.

A case is one site problem (or chain) of a seeded quantum-chemistry Hamiltonian at half filling: L
orbitals, bond dimension about M, TwoU1 or SU2U1.  The MPS is random, with every sector the total
charge allows and sizes in proportion to the states a sector can hold, left-normalised up to the
middle two-site problem and right-normalised after it; the boundaries are grown on the device.

kinds
  hpsi      one H*psi of the middle two-site problem on device vectors (a Davidson iteration's
            operator application; HpsiPlan.apply_device)
  host      the same on host vectors (HpsiPlan.apply), as host-side eigensolvers call it
  davidson  the lowest eigenpair of the middle two-site problem from the MPS's own two-site tensor
            (HpsiPlan.davidson), what every step of a two-site sweep runs
  batch     the lowest eigenpairs of n independent problems in lock step (HpsiPlanBatch.davidson)
  expval    <psi|H|psi> of the chain: L left growth steps (rdm.expval)
  gradient  dE/dh and dE/d(pq|rs) of the chain (adjoint.energy_gradient): right growth steps, left
            growth steps, site plans and their MPO-term gradients

Sizes: 8 to 20 orbitals and bond dimensions of a few dozen up to 2048, the range between the
eight-orbital test problem and the sector sizes (about 80) of the 40-orbital benchmark.  Ragged
sector sizes come by themselves from the proportional bond indices.
"""
import math

import numpy as np
import torch

from qcmaquis_amd import abi
from qcmaquis_amd.adjoint import energy_gradient
from qcmaquis_amd.dmrg import (allowed_bonds, allowed_bonds_su2, left_normalize, merge_two, right_normalize,
                               twosite_offsets)
from qcmaquis_amd.engine import Context, DeviceBoundary, DeviceMPO, DeviceMPS, HpsiPlan, HpsiPlanBatch, lstep, rstep
from qcmaquis_amd.model import Index, MPSLayout
from qcmaquis_amd.qc import QCHamiltonian, make_integrals
from qcmaquis_amd.rdm import expval

SYM = {"2u1": abi.MQ_SYM_TWOU1, "su2": abi.MQ_SYM_SU2U1}
PREC = {"f64": abi.MQ_PREC_FP64, "f32": abi.MQ_PREC_FP32}
DEVICE = "cuda"


def _case(name, kind, sym, L, M, prec="f64", iters=0, n=1):
    c = {"kind": kind, "sym": sym, "L": L, "M": M, "prec": prec, "iters": iters, "n": n}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the eight-orbital test problem: a handful of 1..6-wide tiles, all latency and launches
        _case("hpsi_tiny", "hpsi", "2u1", 8, 40),
        # an edge-of-sweep sized problem called with host vectors, transfers included
        _case("host_small", "host", "2u1", 12, 96),
        # many orbitals at a small bond dimension: millions of MPO terms on tiles of a few elements
        _case("hpsi_small_tiles", "hpsi", "2u1", 18, 128),
        # the bond dimension of production TwoU1 sweeps, odd size
        _case("hpsi_2u1", "hpsi", "2u1", 18, 509),
        # spin-adapted site problem of a mid-sized active space
        _case("hpsi_su2", "hpsi", "su2", 20, 700),
        # spin-adapted, the sector sizes of the M = 2048 benchmark: intermediates of tens of GB
        _case("hpsi_su2_large", "hpsi", "su2", 20, 2048),
        # FP32 contraction of a mixed-precision Davidson, ordinary and large
        _case("hpsi_f32", "hpsi", "2u1", 14, 300, "f32"),
        _case("hpsi_f32_large", "hpsi", "2u1", 18, 512, "f32"),
        # one site solve of a sweep: upload, eight H*psi with their vector operations, download
        _case("davidson", "davidson", "2u1", 14, 256, iters=8),
        # many small independent problems solved together
        _case("batch", "batch", "2u1", 11, 128, iters=4, n=6),
        # an expectation value: one growth step per site, schedules included
        _case("expval", "expval", "2u1", 14, 256),
        # all integral derivatives of a spin-adapted state
        _case("gradient", "gradient", "su2", 12, 200),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["hpsi", "hpsi", "hpsi", "hpsi", "host", "davidson", "batch", "expval", "gradient"])
    if kind == "hpsi":
        if rng.random() < 0.4:
            return _case(None, kind, "su2", rng.randint(12, 20), _log(rng, 60, 2000))
        return _case(None, kind, "2u1", rng.randint(8, 18), _log(rng, 30, 512), rng.choice(["f64", "f64", "f32"]))
    if kind == "host":
        return _case(None, kind, "2u1", rng.randint(8, 14), _log(rng, 30, 300))
    if kind == "davidson":
        sym = rng.choice(["2u1", "su2"])
        return _case(None, kind, sym, rng.randint(8, 16), _log(rng, 30, 400), iters=rng.randint(4, 8))
    if kind == "batch":
        return _case(None, kind, "2u1", rng.randint(8, 12), _log(rng, 40, 200), iters=rng.randint(2, 5), n=rng.randint(2, 6))
    if kind == "expval":
        return _case(None, kind, rng.choice(["2u1", "su2"]), rng.randint(8, 14), _log(rng, 30, 250))
    return _case(None, kind, "su2", rng.randint(8, 12), _log(rng, 30, 190))


# ---- inputs ---------------------------------------------------------------------------------------
_contexts = {}


def _context(sym):
    """one context per symmetry for the process, as a user's program holds it"""
    if sym not in _contexts:
        _contexts[sym] = Context(0, SYM[sym])
    return _contexts[sym]


def _chain(sym, L, M, seed, gradient=False):
    """(Hamiltonian, site layouts, site tensors): integrals and a random MPS from the seed, the MPS
    normalised towards the middle two-site problem (sites L/2-1, L/2)"""
    h, eri, ec = make_integrals(L, seed, 16)
    ham = QCHamiltonian(h, eri, ec, symmetry=SYM[sym], gradient_layout=gradient)
    phys = ham.phys()
    if sym == "su2":
        full = allowed_bonds_su2([phys] * L, (L - L % 2, 0), 1 << 40)
    else:
        full = allowed_bonds([phys] * L, ((L + 1) // 2, L // 2), 1 << 40)
    bonds = []
    for b in full:
        sizes = np.array(b.sizes, np.float64)
        if sizes.sum() > M:
            sizes = np.maximum(1.0, np.floor(sizes * M / sizes.sum()))
        bonds.append(Index(b.charges, [int(x) for x in sizes]))
    lay = [MPSLayout(bonds[k], phys, bonds[k + 1]) for k in range(L)]
    rng = np.random.default_rng(seed)
    data = [rng.standard_normal(x.n) for x in lay]
    mid = L // 2 - 1
    left_normalize(lay, data, mid)
    right_normalize(lay, data, stop=mid + 2)
    for k in (mid, mid + 1):
        data[k] = data[k] / np.linalg.norm(data[k])
    return ham, lay, data


def _site_vector(sym, ham, lay, data, seed):
    """layout of the middle two-site problem and a normalised vector on it: the MPS's two-site
    tensor (TwoU1) or a random vector of the pair-coupled basis (SU2U1)"""
    L = len(lay)
    mid = L // 2 - 1
    phys2 = ham.phys(True)
    if sym == "su2":
        lay2 = MPSLayout(lay[mid].left, phys2, lay[mid + 1].right)
        psi = np.random.default_rng([seed, 1]).standard_normal(lay2.n)
    else:
        lay2, psi = merge_two(lay[mid], data[mid], lay[mid + 1], data[mid + 1], phys2, twosite_offsets(ham.phys()))
    return lay2, psi / np.linalg.norm(psi)


def _problem(ctx, sym, L, M, seed):
    """(two-site MPO, left boundary, right boundary, layout) of the middle site problem, its vector"""
    ham, lay, data = _chain(sym, L, M, seed)
    mid = L // 2 - 1
    left = DeviceBoundary.initial(ctx, lay[0].left, ham.mpo(0).row_dim)
    for k in range(mid):
        m = DeviceMPS(ctx, lay[k], data[k])
        left = lstep(ctx, DeviceMPO(ctx, ham.mpo(k)), left, m, m)
    right = DeviceBoundary.initial(ctx, lay[-1].right, ham.mpo(L - 1).col_dim)
    for k in range(L - 1, mid + 1, -1):
        m = DeviceMPS(ctx, lay[k], data[k])
        right = rstep(ctx, DeviceMPO(ctx, ham.mpo(k)), right, m, m)
    lay2, psi = _site_vector(sym, ham, lay, data, seed)
    return (DeviceMPO(ctx, ham.mpo(mid, True)), left, right, lay2), psi


def prepare(case, seed):
    sym, L, M, kind = case["sym"], case["L"], case["M"], case["kind"]
    ctx = _context(sym)
    st = {"case": case, "ctx": ctx}
    if kind in ("expval", "gradient"):
        ham, lay, data = _chain(sym, L, M, seed, gradient=kind == "gradient")
        st.update(ham=ham, lay=lay, data=data)
        return st
    if kind == "batch":
        made = [_problem(ctx, sym, L - i % 3, M, seed * 64 + i) for i in range(case["n"])]
        st.update(plan=HpsiPlanBatch(ctx, [m[0] for m in made]), psi=[m[1] for m in made])
        return st
    item, psi = _problem(ctx, sym, L, M, seed)
    st.update(plan=HpsiPlan(ctx, *item), item=item, psi=psi)
    if kind == "hpsi":
        x = torch.from_numpy(psi).to(DEVICE)
        st.update(x=x, y=torch.empty_like(x))
        torch.cuda.synchronize()
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind, prec = case["kind"], PREC[case["prec"]]
    if kind == "hpsi":
        st["plan"].apply_device(st["x"].data_ptr(), st["y"].data_ptr(), prec)
        return st["y"]
    if kind == "host":
        return st["plan"].apply(st["psi"], prec)
    if kind == "davidson":
        e, v, _ = st["plan"].davidson(st["psi"], tol=1e-12, max_iter=case["iters"], precision=prec)
        return {"e": e, "v": v}
    if kind == "batch":
        e, v, _, _ = st["plan"].davidson(st["psi"], tol=1e-12, max_iter=case["iters"], precision=prec)
        return {"e": e, "v": v}
    if kind == "expval":
        return expval(ctx, st["lay"], st["data"], st["ham"])
    e, dh, deri, _ = energy_gradient(ctx, st["ham"], st["lay"], st["data"])
    return {"e": e, "dh": dh, "deri": deri}


def work(case):
    """flops: the T products, the MPO-term sum and the output products of every contraction (two per
    multiply-add, each MPO term once); bytes: every boundary read or written, the site tensors and
    vectors, in the precision of the contraction"""
    sym, L, M, kind = case["sym"], case["L"], case["M"], case["kind"]
    ctx = _context(sym)
    if kind in ("expval", "gradient"):
        ham, lay, data = _chain(sym, L, M, 1, gradient=kind == "gradient")
        flops = size = 0
        b = DeviceBoundary.initial(ctx, lay[0].left, ham.mpo(0).row_dim)
        for k in range(L):
            m = DeviceMPS(ctx, lay[k], data[k])
            b = lstep(ctx, DeviceMPO(ctx, ham.mpo(k)), b, m, m)
            g = b.growth_stats()
            flops += g["flops_total"]
            size += 8 * (2 * g["out_elements"] + lay[k].n)
        # the gradient grows both boundary chains and forms one more contraction of every site
        return {"bytes": 3 * size, "flops": 3 * flops} if kind == "gradient" else {"bytes": size, "flops": flops}
    if kind == "batch":
        made = [_problem(ctx, sym, L - i % 3, M, 64 + i) for i in range(case["n"])]
        s = HpsiPlanBatch(ctx, [m[0] for m in made]).stats()
    else:
        s = HpsiPlan(ctx, *_problem(ctx, sym, L, M, 1)[0]).stats()
    reps = case["iters"] or 1
    vec = 16 * s["psi_elements"]
    size = s["bytes_compulsory"] - vec
    return {"bytes": reps * (size // (2 if case["prec"] == "f32" else 1) + vec), "flops": reps * s["flops_total"]}


# ---- 64-bit values in plain torch (TwoU1) ---------------------------------------------------------
# Every MPO index b of a TwoU1 chain carries one charge q_b, and a boundary maps ket sector c to bra
# sector c + q_b: it is held as {ket sector: {q: tensor (indices of charge q, bra size, ket size)}}
# over all indices of the charge, absent blocks being zero.  Each contraction is dense over the
# indices of a charge.
def _states(phys):
    return [(c, i) for c, d in zip(phys.charges, phys.sizes) for i in range(d)]


class _Site:
    """one MPO tensor: w[s'] is the (row index) x (ket state s, column index) matrix of the entries"""

    def __init__(self, mpo, phys):
        spec = mpo.to_spec()
        st = _states(phys)
        pos = {x: i for i, x in enumerate(st)}
        self.charge = [c for c, _ in st]
        self.n, self.rows, self.cols = len(st), spec.row_dim, spec.col_dim
        acc = {}
        for (b1, b2), terms in spec.terms.items():
            for op, scale in terms:
                for ci, co, entries in spec.ops[op].blocks:
                    for e in entries:
                        i, o = pos.get((tuple(ci), e[0])), pos.get((tuple(co), e[1]))
                        if i is not None and o is not None:
                            acc[o, b1, i, b2] = acc.get((o, b1, i, b2), 0.0) + scale * e[2]
        key = np.array(list(acc), np.int64).reshape(-1, 4)
        self.key = key
        w = torch.zeros(self.n, self.rows, self.n, self.cols, dtype=torch.float64, device=DEVICE)
        k = torch.from_numpy(key).to(DEVICE)
        w[k[:, 0], k[:, 1], k[:, 2], k[:, 3]] = torch.tensor(list(acc.values()), dtype=torch.float64, device=DEVICE)
        self.w = w

    def column_charges(self, rows):
        """charges of the column indices from those of the row indices (bra minus ket charge)"""
        out = [None] * self.cols
        for o, b1, i, b2 in self.key:
            a, b = self.charge[o], self.charge[i]
            out[b2] = (rows[b1][0] + a[0] - b[0], rows[b1][1] + a[1] - b[1])
        return out


def _groups(charges):
    """{charge: its indices on the device}"""
    g = {}
    for i, q in enumerate(charges):
        if q is not None:
            g.setdefault(q, []).append(i)
    return {q: torch.tensor(v, device=DEVICE) for q, v in g.items()}


def _add(a, b):
    return (a[0] + b[0], a[1] + b[1])


def _sub(a, b):
    return (a[0] - b[0], a[1] - b[1])


def _blocks(lay, data):
    """{(left charge, state): block} of a right-paired site tensor, on the device"""
    out = {}
    for li, lc in enumerate(lay.left.charges):
        m = torch.from_numpy(np.ascontiguousarray(lay.rp_block(data, li))).to(DEVICE)
        for s, (c, i) in enumerate(_states(lay.phys)):
            rc = _add(lc, c)
            if rc in lay.right.charges:
                rs = lay.right.size_of(rc)
                o = lay.rpb[(c, rc)] + i * rs
                out[lc, s] = m[:, o:o + rs].contiguous()
    return out


def _grow_left(site, gl, gr, left, lay, data):
    """boundary right of the site: L'_b2 = sum A^T L_b1 W A"""
    blk = _blocks(lay, data)
    wt = site.w.permute(0, 3, 2, 1).contiguous()  # [s'][b2][s][b1]
    out = {}
    for (lb, o), bra in blk.items():
        rb = _add(lb, site.charge[o])
        for rc in lay.right.charges:
            q2 = _sub(rb, rc)
            if q2 not in gr:
                continue
            t, w = [], []
            for i in range(site.n):
                lc = _sub(rc, site.charge[i])
                q1 = _sub(lb, lc)
                if (lc, i) in blk and lc in left and q1 in left[lc]:
                    t.append((left[lc][q1] @ blk[lc, i]).flatten(1))
                    w.append(wt[o][gr[q2], i][:, gl[q1]])
            if t:
                s = (torch.cat(w, 1) @ torch.cat(t, 0)).view(len(gr[q2]), bra.shape[0], -1)
                v = bra.t().contiguous() @ s
                d = out.setdefault(rc, {})
                d[q2] = d[q2] + v if q2 in d else v
    return out


def _grow_right(site, gl, gr, right, lay, data):
    """boundary left of the site: R_b1 = sum A W R_b2 A^T, blocks held ket size x bra size"""
    blk = _blocks(lay, data)
    out = {}
    for (lb, o), bra in blk.items():
        rb = _add(lb, site.charge[o])
        for lc in lay.left.charges:
            q1 = _sub(lb, lc)
            if q1 not in gl:
                continue
            s = _rows(site, gl, gr, right, blk, lc, rb, o, q1)
            if s is not None:
                v = s @ bra.t().contiguous()
                d = out.setdefault(lc, {})
                d[q1] = d[q1] + v if q1 in d else v
    return out


def _rows(site, gl, gr, right, blk, lc, rb, o, q1, cache=None):
    """S_b1 = sum W psi R_b2 over the ket states, for the ket sector lc and the bra state o -> rb"""
    t, w = [], []
    for i in range(site.n):
        if (lc, i) not in blk:
            continue
        rc = _add(lc, site.charge[i])
        q2 = _sub(rb, rc)
        if rc in right and q2 in right[rc]:
            if cache is None:
                t.append((blk[lc, i] @ right[rc][q2]).flatten(1))
            else:
                if (lc, i, rb) not in cache:
                    cache[lc, i, rb] = (blk[lc, i] @ right[rc][q2]).flatten(1)
                t.append(cache[lc, i, rb])
            w.append(site.w[o][gl[q1], i][:, gr[q2]])
    if not t:
        return None
    ls = next(x.shape[0] for (c, _), x in blk.items() if c == lc)
    return (torch.cat(w, 1) @ torch.cat(t, 0)).view(len(gl[q1]), ls, -1)


def _ones(index):
    return {c: {(0, 0): torch.ones(1, s, s, dtype=torch.float64, device=DEVICE)} for c, s in zip(index.charges, index.sizes)}


def _exact_hpsi(L, M, seed):
    ham, lay, data = _chain("2u1", L, M, seed)
    mid = L // 2 - 1
    phys = ham.phys()
    sites = [_Site(ham.mpo(k), phys) for k in range(L)]
    charges = [[(0, 0)] * sites[0].rows]
    for s in sites:
        charges.append(s.column_charges(charges[-1]))
    groups = [_groups(q) for q in charges]
    left, right = _ones(lay[0].left), _ones(lay[-1].right)
    for k in range(mid):
        left = _grow_left(sites[k], groups[k], groups[k + 1], left, lay[k], data[k])
    for k in range(L - 1, mid + 1, -1):
        right = _grow_right(sites[k], groups[k], groups[k + 1], right, lay[k], data[k])
    lay2, psi = _site_vector("2u1", ham, lay, data, seed)
    del sites
    site = _Site(ham.mpo(mid, True), lay2.phys)
    gl, gr = groups[mid], groups[mid + 2]
    blk = _blocks(lay2, psi)
    out = np.zeros(lay2.n)
    # bra right sectors one after the other: the products psi R of one sector are kept, then dropped
    for rb in lay2.right.charges:
        cache = {}
        for o, (c, i) in enumerate(_states(lay2.phys)):
            lb = _sub(rb, c)
            if lb not in lay2.left.charges:
                continue
            y = None
            for lc in lay2.left.charges:
                q1 = _sub(lb, lc)
                if lc not in left or q1 not in left[lc]:
                    continue
                s = _rows(site, gl, gr, right, blk, lc, rb, o, q1, cache)
                if s is not None:
                    a = left[lc][q1].permute(1, 0, 2).flatten(1)
                    v = a @ s.flatten(0, 1)
                    y = v if y is None else y + v
            if y is not None:
                li = lay2.left.position(lb)
                col = lay2.rpb[(c, rb)] + i * y.shape[1]
                lay2.rp_block(out, li)[:, col:col + y.shape[1]] = y.cpu().numpy()
    return out


def _exact_expval(L, M, seed):
    ham, lay, data = _chain("2u1", L, M, seed)
    q, b = [(0, 0)], _ones(lay[0].left)
    for k in range(L):
        site = _Site(ham.mpo(k), ham.phys())
        nq = site.column_charges(q)
        b = _grow_left(site, _groups(q), _groups(nq), b, lay[k], data[k])
        q = nq
    (d,) = b.values()
    return float(d[(0, 0)].item())


def exact(case, seed):
    if case["sym"] != "2u1":
        return None  # spin-adapted: the coupling coefficients exist in this package only
    if case["kind"] in ("hpsi", "host"):
        return _exact_hpsi(case["L"], case["M"], seed)
    if case["kind"] == "expval":
        return _exact_expval(case["L"], case["M"], seed)
    return None  # a fixed number of Davidson iterations: no closed form
