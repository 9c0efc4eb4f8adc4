"""The work whose time counts: calls that DMRG, VUMPS and TDVP programs make of
this library, from the latency-bound pivots to the ones that fill the card.

A case names a `kind` of call, the model whose MPO and bond sectors it uses,
the bond dimension M and the number `nleft` of sites left of the pivot:

  hxv            one effective-Hamiltonian application on device vectors
                 (vmps_hxv_device), or with `host` on host arrays (HxV, the
                 call the drop-in adapter serves); `n` > 1 pivots as one batch
  lanczos        the lowest eigenpair of a pivot from a start vector on the
                 device, in FP64 or mixed precision with FP64 refinement
  lanczos_batch  one eigenpair for each of `n` pivots, solved together
  advance        the sweep moves one site on: contract_L on the device, the
                 plan of the next pivot, one HxV on it

Environments are made as a sweep in canonical gauge meets them: the channel
of the MPO that has not started an operator string carries the identity, the
finished one the block Hamiltonian (here levels plus a random perturbation),
the open channels random operators of norm about one.
"""
import ctypes
import functools
import math
from fractions import Fraction

import numpy as np
import torch

from vmps_amd import _lib, env, lattice, models, synth
from vmps_amd.pivot import DeviceVector, HxV, PivotBatch, PivotMatrix1, PivotMatrix2, lanczos_batch, lanczos_device

CLASSES = {1: PivotMatrix1, 2: PivotMatrix2}
TUNE_MIN_FLOPS = 1e9  # pivots of at least this work get autotuned tiles, as dmrg.GpuBackend has it
TOL = dict(tol_eigval=1e-12, tol_state=1e-10)
MAX_ITER = 200
TYPICAL_HXV = 100  # HxV applications of a solve to TOL, measured: 70 to 180


def listed():
    return [
        # the smallest call: an HxV of a short U(1) chain, two launches
        dict(name="hxv_heisenberg_M64", kind="hxv", model="heisenberg", M=64, nleft=15, nsite=2, prec="fp64", n=1,
             host=False),
        # a Hubbard chain at moderate M: over a hundred sectors, blocks of a few rows
        dict(name="hxv_hubbard_M512", kind="hxv", model="hubbard", M=512, nleft=23, nsite=2, prec="fp64", n=1,
             host=False),
        # one-site HxV (VUMPS, TDVP) through the host-buffer call of the drop-in adapter
        dict(name="hxv1_host_hubbard_M512", kind="hxv", model="hubbard", M=512, nleft=23, nsite=1, prec="fp64", n=1,
             host=True),
        # a production U(1) chain: blocks of one to three hundred rows
        dict(name="hxv_heisenberg_M2048", kind="hxv", model="heisenberg", M=2048, nleft=31, nsite=2, prec="fp64", n=1,
             host=False),
        # spin SU(2) x charge U(1) ladder in FP32, blocks up to about 120 rows
        dict(name="hxv_fp32_ladder_M2048", kind="hxv", model="ladder", M=2048, nleft=31, nsite=2, prec="fp32", n=1,
             host=False),
        # the headline model: C60 Heisenberg SU(2) at M = 4096, the plain FP64 product ...
        dict(name="hxv_c60_M4096", kind="hxv", model="c60", M=4096, nleft=29, nsite=2, prec="fp64", n=1, host=False),
        # ... and the split-BF16 one, in which a mixed solve spends its time
        dict(name="hxv_bf16_c60_M4096", kind="hxv", model="c60", M=4096, nleft=29, nsite=2, prec="bf16x3", n=1,
             host=False),
        # the sites of a VUMPS cell at once: independent pivots of many sizes in one plan
        dict(name="hxv_batch16", kind="hxv", model="mixture", M=1024, nleft=20, nsite=2, prec="fp64", n=16,
             host=False),
        # a whole eigensolve on the Hubbard pivot: HxV, Gram-Schmidt and the host's part of the iteration
        dict(name="lanczos_hubbard_M512", kind="lanczos", model="hubbard", M=512, nleft=23, nsite=2, prec="fp64", n=1),
        # a mixed solve: split-BF16 Lanczos, conjugate-gradient corrections, FP64 residuals
        dict(name="lanczos_mixed_heisenberg_M2048", kind="lanczos", model="heisenberg", M=2048, nleft=31, nsite=2,
             prec="bf16x3", n=1),
        # the eigensolves of a VUMPS cell together
        dict(name="lanczos_batch8", kind="lanczos_batch", model="mixture", M=256, nleft=20, nsite=2, prec="fp64", n=8),
        # one step along the chain: environment update, plan of the next pivot, its first HxV
        dict(name="advance_heisenberg_M1024", kind="advance", model="heisenberg", M=1024, nleft=20, nsite=2,
             prec="fp64", n=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hxv", "hxv", "hxv", "hxv", "batch", "lanczos", "lanczos_batch", "advance"])
    nleft = rng.randrange(12, 40)
    if kind == "hxv":
        model, lo, hi = rng.choice([("heisenberg", 32, 2048), ("hubbard", 64, 1024), ("ladder", 256, 2048),
                                    ("c60", 256, 4096)])
        nsite = rng.choice([1, 2, 2, 2]) if model in ("heisenberg", "hubbard") else 2
        prec = rng.choice(["fp64", "fp64", "fp32", "bf16x3", "bf16x3"])
        M = _log_int(rng, lo, hi)
        return dict(kind="hxv", model=model, M=M, nleft=nleft, nsite=nsite, prec=prec, n=1,
                    host=M <= 1024 and rng.random() < 0.2)
    if kind == "batch":
        return dict(kind="hxv", model="mixture", M=_log_int(rng, 64, 1024), nleft=nleft, nsite=2,
                    prec=rng.choice(["fp64", "bf16x3"]), n=rng.randrange(2, 17), host=False)
    if kind == "lanczos":
        model, lo, hi = rng.choice([("heisenberg", 64, 2048), ("hubbard", 64, 512)])
        return dict(kind="lanczos", model=model, M=_log_int(rng, lo, hi), nleft=nleft, nsite=2,
                    prec=rng.choice(["fp64", "bf16x3"]), n=1)
    if kind == "lanczos_batch":
        return dict(kind="lanczos_batch", model="mixture", M=_log_int(rng, 64, 256), nleft=nleft, nsite=2, prec="fp64",
                    n=rng.randrange(2, 9))
    return dict(kind="advance", model=rng.choice(["heisenberg", "hubbard"]), M=_log_int(rng, 64, 1024), nleft=nleft,
                nsite=2, prec="fp64", n=1)


# ---- pivots -----------------------------------------------------------------
def _site(model, l):
    if model == "heisenberg":
        return models.heisenberg_u1_mpo()
    if model == "hubbard":
        return models.hubbard_u1xu1_mpo(t=1.0, U=8.0)
    if model == "ladder":
        return models.hubbard_su2xu1_ladder_mpo(t=1.0, U=6.0, rung=l % 2 == 0)
    return _c60_sites()[l]


@functools.lru_cache(maxsize=1)
def _c60_sites():
    return models.heisenberg_su2_full_mpo(lattice.c60_couplings())


@functools.lru_cache(maxsize=None)
def _bond(model, l, M, tail):
    if model == "heisenberg":
        return synth.heisenberg_bond(l, M)
    if model == "hubbard" and tail:
        # many sectors of one or two states, a few of tens: synth.hubbard_bond's
        # profile of an odd bond, whose centre (N odd, 2Sz = 0) is no sector itself
        allowed = [(n, s) for n in range(2 * l + 1) for s in range(-l, l + 1)
                   if (n - s) % 2 == 0 and abs(s) <= min(n, 2 * l - n)]
        return synth.stretched_sectors((l | 1, 0), M, 0.36, 0.02, allowed)
    if model == "hubbard":
        return synth.hubbard_bond(l, M, alpha=1.0, lam=2.2)
    if model == "ladder":
        return synth.hubbard_su2xu1_bond(l, M, filling=0.875)
    return synth.heisenberg_su2_bond(l, M)


def _layout(sym, aux, bond, left):
    """Sectors (qin, qout, qmid, rows, cols, channels) of an environment over `bond`."""
    dim, out = dict(bond), []
    for qmid, channels in aux:
        for q, d in bond:
            for p in sym.reduce(q, qmid):
                if p in dim:
                    out.append((p, q, tuple(qmid), dim[p], d, channels) if left
                               else (q, p, tuple(qmid), d, dim[p], channels))
    return out


def _levels(bond):
    """Energies of the states of each sector: lowest near the bond's mean charge."""
    centre = np.average(np.array([q for q, _ in bond], float), axis=0, weights=[d for _, d in bond])
    return {q: min(2.0, 0.15 * float(np.sum((np.array(q) - centre) ** 2))) + 2.5 * np.sqrt(np.arange(d) / d)
            for q, d in bond}


def _environment(W, bond, left, rng):
    """L over `bond` with W's incoming channels, or R with its outgoing ones."""
    sym, aux, conj = W.sym, W.aux_in if left else W.aux_out, W.conj_in if left else W.conj_out
    lay = _layout(sym, aux, bond, left)
    data = rng.standard_normal(sum(r * c * n for (_, _, _, r, c, n) in lay))
    first, g = {}, 0
    for q, n in aux:
        first[tuple(q)] = g
        g += n
    owner = [(tuple(q), a) for q, n in aux for a in range(n)]
    sectors, index, off = [], {}, 0
    for qin, qout, qmid, r, c, n in lay:
        blocks = []
        for _ in range(n):
            blocks.append(data[off:off + r * c].reshape((r, c), order="F"))
            off += r * c
        index[(qin, qout, qmid)] = blocks
        sectors.append((qin, qout, qmid, blocks))
    level = _levels(bond)
    vac = sym.vacuum()
    n_vac = dict((tuple(q), n) for q, n in aux)[vac]
    identity, energy = (n_vac - 1, 0) if left else (0, n_vac - 1)
    for qin, qout, qmid, blocks in sectors:
        for a, x in enumerate(blocks):
            x *= 0.5 / math.sqrt(max(x.shape))
            if qmid == vac and a == identity:
                x[...] = np.eye(*x.shape)
            elif qmid == vac and a == energy:
                x *= 0.2
                x[np.diag_indices(x.shape[0])] += level[qin]
    if conj is not None:  # a Hermitian H: the transposed operator string's block is the transpose
        done = set()
        for qin, qout, qmid, blocks in sectors:
            for a, x in enumerate(blocks):
                qc, ac = owner[conj[first[qmid] + a]]
                if (qout, qin, qc, ac) in done:
                    continue
                done.add((qin, qout, qmid, a))
                y = index[(qout, qin, qc)][ac]
                if y is x:
                    x[...] = 0.5 * (x + x.T)
                else:
                    y[...] = x.T
    return sectors


def _shape(W12, W34, left, right):
    """A pivot without its environments."""
    pd = synth.PivotData(W12.sym, W12, W34, left, right, nsite=2 if W34 else 1)
    rdim = dict(right)
    if W34 is None:
        pd.basis = [(tuple(q), s) for s, q in enumerate(W12.qloc)]
    else:
        pd.basis = synth.two_site_basis(W12.sym, W12.qloc, W34.qloc)
    for b in pd.basis:
        pd.V.append([(qin, tuple(qout), d, rdim[qout]) for qin, d in left for qout in W12.sym.reduce(qin, b[0])
                     if qout in rdim])
    return pd


def _shapes(case):
    """The case's pivots, layout only."""
    if case["model"] != "mixture":
        model, l, ns, M = case["model"], case["nleft"], case["nsite"], case["M"]
        return [_shape(_site(model, l), _site(model, l + 1) if ns == 2 else None, _bond(model, l, M, True),
                       _bond(model, l + ns, M, True))]
    out = []
    for i in range(case["n"]):  # Heisenberg and Hubbard sites in turn, M falling to an eighth of the largest
        model, l = ("heisenberg", "hubbard")[i % 2], case["nleft"] + i % 5
        M = max(8, int(case["M"] * 8.0 ** (-i / max(1, case["n"] - 1))))
        W = _site(model, l)
        out.append(_shape(W, W, _bond(model, l, M, False), _bond(model, l + 2, M, False)))
    return out


def _pivots(case, rng):
    out = _shapes(case)
    for pd in out:
        pd.L = _environment(pd.W12, pd.left, True, rng)
        pd.R = _environment(pd.W34 or pd.W12, pd.right, False, rng)
    return out


def _vector(pds, rng):
    """A wavefunction as a sweep hands it over: weight falling with the energies of
    the bond states, with noise on every element."""
    out = []
    for pd in pds:
        left, right = _levels(pd.left), _levels(pd.right)
        v = rng.standard_normal(pd.vsize) * 0.2
        for _, qin, qout, off, r, c in pd.block_offsets():
            weight = np.exp(-1.5 * (left[qin][None, :] + right[qout][:, None]))  # [column, row]
            v[off:off + r * c] = ((1.0 + v[off:off + r * c].reshape(c, r)) * weight).ravel()
        out.append(v / np.linalg.norm(v))
    return np.concatenate(out)


def _advance(case, rng):
    """Old left environment, site tensor A (column-orthonormal up to rounding of a
    random matrix) and the pivot one site further right, without its L."""
    model, l, M = case["model"], case["nleft"], case["M"]
    W = _site(model, l)
    left, mid, right = (_bond(model, l + k, M, True) for k in (0, 1, 3))
    old = _environment(W, left, True, rng)
    mdim = dict(mid)
    A = [[(qin, qout, np.asfortranarray(rng.standard_normal((d, mdim[qout])) / math.sqrt(len(W.qloc) * d)))
          for qin, d in left for qout in W.sym.reduce(qin, q) if qout in mdim] for q in W.qloc]
    pd = _shape(W, W, mid, right)
    pd.R = _environment(W, right, False, rng)
    return W, left, old, A, pd


# ---- the calls ----------------------------------------------------------------
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "advance":
        W, left, old, A, pd = _advance(case, rng)
        nq = W.sym.nq
        pd.R = env.DeviceEnv.from_host(pd.R, nq)
        vin = torch.from_numpy(_vector([pd], rng)).cuda()
        torch.cuda.synchronize()
        return dict(kind=kind, W=W, old=env.DeviceEnv.from_host(old, nq), A=A, pd=pd, vin=vin)
    pds = _pivots(case, rng)
    if case["model"] == "mixture":
        H = PivotBatch(pds, precision=case["prec"])
    else:
        H = CLASSES[case["nsite"]](pds[0], precision=case["prec"])
    if H.stats()["flops_alg"] >= TUNE_MIN_FLOPS:
        H.autotune(iters=3)
    for pd in pds:
        pd.L = pd.R = None
    state = dict(kind=kind, H=H, prec=case["prec"], host=case.get("host", False))
    v = _vector(pds, rng)
    if kind == "lanczos_batch" or state["host"]:
        state["vin"] = v
    else:
        state["vin"] = torch.from_numpy(v).cuda()
        state["vout"] = torch.empty_like(state["vin"])
    if kind == "lanczos":
        state["dv"] = DeviceVector(H)
        state["start"] = v
    torch.cuda.synchronize()
    return state


def _hxv_device(H, vin, vout):
    _lib.check(H._lib.vmps_hxv_device(H._plan, ctypes.c_void_p(vin.data_ptr()), ctypes.c_void_p(vout.data_ptr()), None))
    return vout


def run(state):
    kind = state["kind"]
    if kind == "hxv":
        if state["host"]:
            return HxV(state["H"], state["vin"])
        return _hxv_device(state["H"], state["vin"], state["vout"])
    if kind == "lanczos":
        dv = state["dv"]
        dv.upload(state["start"])
        r = lanczos_device(state["H"], dv, precision=state["prec"], max_iter=MAX_ITER, refine_tol_eigval=TOL["tol_eigval"],
                           refine_tol_state=TOL["tol_state"], **TOL)
        return dict(energy=r["energy"], vector=dv.download())
    if kind == "lanczos_batch":
        v, res = lanczos_batch(state["H"], v0=state["vin"], max_iter=MAX_ITER, **TOL)
        return dict(energies=np.array([r["energy"] for r in res]), vector=v)
    pd = state["pd"]
    pd.L = env.contract_L(state["W"], state["old"], state["A"], state["A"], device=True)
    H = PivotMatrix2(pd)
    vout = torch.empty_like(state["vin"])
    _hxv_device(H, state["vin"], vout)
    H.close()
    pd.L.close()
    return vout


# ---- 64-bit results and work, from the definitions -----------------------------
@functools.lru_cache(maxsize=None)
def _six_j(a, b, c, d, e, f):
    """Wigner 6j of spins a/2 .. f/2, Racah's formula in exact fractions."""
    triads = ((a, b, c), (a, e, f), (d, b, f), (d, e, c))
    for x, y, z in triads:
        if (x + y + z) % 2 or not abs(x - y) <= z <= x + y:
            return 0.0
    fac = math.factorial
    norm = Fraction(1)
    for x, y, z in triads:
        norm *= Fraction(fac((x + y - z) // 2) * fac((x - y + z) // 2) * fac((y + z - x) // 2),
                         fac((x + y + z) // 2 + 1))
    t = [sum(x) // 2 for x in triads]
    u = [(a + b + d + e) // 2, (b + c + e + f) // 2, (a + c + d + f) // 2]
    total = 0
    for z in range(max(t), min(u) + 1):
        den = 1
        for x in t:
            den *= fac(z - x)
        for x in u:
            den *= fac(x - z)
        total += Fraction((-1) ** z * fac(z + 1), den)
    return math.copysign(math.sqrt(norm * total * total), total) if total else 0.0


@functools.lru_cache(maxsize=None)
def _nine(q):
    """sqrt(q7 q8 q3 q6) times the 9j symbol of spins (q_i - 1) / 2."""
    a, b, c, d, e, f, g, h, i = (x - 1 for x in q)
    lo, hi = max(abs(a - i), abs(d - h), abs(b - f)), min(a + i, d + h, b + f)
    s = sum((-1) ** x * (x + 1) * _six_j(a, d, g, h, i, x) * _six_j(b, e, h, d, x, f) * _six_j(c, f, i, x, a, b)
            for x in range(lo, hi + 1, 2))
    return s * math.sqrt(q[6] * q[7] * q[2] * q[5])


def _recouple(sym, *qs):
    """Product over the SU(2) components of the nine- or six-argument coupling factor."""
    out = 1.0
    for k, kind in enumerate(sym.kinds):
        if kind == models.SU2_KIND:
            q = tuple(x[k] for x in qs)
            if len(q) == 9:
                out *= _nine(q)
            else:
                out *= (_six_j(*(x - 1 for x in q)) * math.sqrt(q[2] * q[5])
                        * (-1) ** ((q[0] + q[1] + q[3] + q[4] - 4) // 2))
    return out


def _transitions(pd):
    """{(component out, in, operator, left mid, right mid): {(a, b): coefficient}} of the pivot's MPO."""
    sym, W1, W2, out = pd.sym, pd.W12, pd.W34, {}

    def put(key, a, b, c):
        if abs(c) > 1e-14:
            d = out.setdefault(key, {})
            d[(a, b)] = d.get((a, b), 0.0) + c

    if pd.nsite == 1:
        for s1, s2, k, qi, qo, _, _, row, col, val in W1.blocks:
            for a, b, c in zip(row, col, val):
                put((s1, s2, tuple(W1.qop[k]), tuple(qi), tuple(qo)), int(a), int(b), float(c))
        return out
    comps = {}
    for s, (qm, s1, s3) in enumerate(pd.basis):
        comps.setdefault((s1, s3), []).append((s, tuple(qm)))
    for s1, s2, k1, qi, qw, _, _, r1, c1, v1 in W1.blocks:
        for s3, s4, k2, qx, qo, _, _, r2, c2, v2 in W2.blocks:
            if tuple(qw) != tuple(qx):
                continue
            pairs = [(a, b, x * y) for a, w, x in zip(r1, c1, v1) for z, b, y in zip(r2, c2, v2) if w == z]
            o1, o2 = tuple(W1.qop[k1]), tuple(W2.qop[k2])
            for op in sym.reduce(o1, o2) if pairs else ():
                six = _recouple(sym, qi, o1, qw, o2, qo, op)
                for so, mo in comps[(s1, s3)]:
                    for si, mi in comps[(s2, s4)]:
                        f = six * _recouple(sym, W1.qloc[s2], W2.qloc[s4], mi, o1, o2, op, W1.qloc[s1], W2.qloc[s3],
                                            mo) if six else 0.0
                        for a, b, x in pairs:
                            put((so, si, tuple(op), tuple(qi), tuple(qo)), int(a), int(b), f * x)
    return out


def _terms(pd):
    """Contributions (out block, L block, in block, R block, coefficient); blocks
    of L and R are (qin, qout, qmid, channel), those of the vector (s, qin, qout)."""
    sym = pd.sym
    ldim, rdim = dict(pd.left), dict(pd.right)
    by_in = [{} for _ in pd.V]
    for s, blocks in enumerate(pd.V):
        for qin, qout, _, _ in blocks:
            by_in[s].setdefault(tuple(qin), []).append(tuple(qout))
    locq = [tuple(b[0]) for b in pd.basis]
    for (so, si, op, lmid, rmid), pairs in _transitions(pd).items():
        for ket in by_in[si]:
            for bra in sym.reduce(ket, lmid):
                if bra not in ldim or bra not in by_in[so]:
                    continue
                for x in by_in[si][ket]:
                    for y in by_in[so][bra]:
                        if x not in rdim or not sym.validate3(x, rmid, y):
                            continue
                        f = _recouple(sym, ket, locq[si], x, lmid, op, rmid, bra, locq[so], y)
                        if abs(f) > 1e-14:
                            for (a, b), c in pairs.items():
                                if abs(c) > 1e-14:
                                    yield (so, bra, y), (bra, ket, lmid, a), (si, ket, x), (x, y, rmid, b), f * c


def _hxv_work(pds):
    flops = byts = 0.0
    for pd in pds:
        ld, rd = dict(pd.left), dict(pd.right)
        t, u, ls, rs = set(), set(), set(), set()
        for o, l, v, r, _ in _terms(pd):
            t.add((l, v))
            u.add((o, r))
            ls.add(l)
            rs.add(r)
        flops += sum(2.0 * ld[l[0]] * ld[l[1]] * rd[v[2]] for l, v in t)
        flops += sum(2.0 * ld[o[1]] * rd[r[0]] * rd[r[1]] for o, r in u)
        byts += 16.0 * pd.vsize + 8.0 * sum(ld[l[0]] * ld[l[1]] for l in ls) + 8.0 * sum(rd[r[0]] * rd[r[1]] for r in rs)
    return byts, flops


def work(case):
    if case["kind"] == "advance":
        # each block of the old L, A, the new L and R once; the products of the two contractions
        W = _site(case["model"], case["nleft"])
        left, mid, right = (_bond(case["model"], case["nleft"] + k, case["M"], True) for k in (0, 1, 3))
        byts, flops = _hxv_work([_shape(W, W, mid, right)])
        ld, md = dict(left), dict(mid)
        old = _layout(W.sym, W.aux_in, left, True)
        byts += 8.0 * sum(r * c * n for (_, _, _, r, c, n) in old)
        byts += 8.0 * sum(ld[q] * md[p] for s in W.qloc for q in ld for p in W.sym.reduce(q, s) if p in md)
        byts += 8.0 * sum(r * c * n for (_, _, _, r, c, n) in _layout(W.sym, W.aux_out, mid, True))
        for qin, qout, _, r, c, n in old:  # L . A_ket, then A_bra^T . (L A)
            for s in W.qloc:
                for p in W.sym.reduce(qout, s):
                    if p in md:
                        flops += 2.0 * n * r * c * md[p]
        for qin, _, _, r, c, n in _layout(W.sym, W.aux_out, mid, True):
            for s in W.qloc:
                flops += 2.0 * n * r * c * sum(d for q, d in left if qin in W.sym.reduce(q, s))
        return dict(bytes=byts, flops=flops)
    byts, flops = _hxv_work(_shapes(case))
    if case["kind"] != "hxv":
        n = sum(pd.vsize for pd in _shapes(case))
        # every application reads its operands; the iteration reads and writes a few vectors beside them
        byts, flops = TYPICAL_HXV * (byts + 8.0 * 6 * n), TYPICAL_HXV * (flops + 12.0 * n)
    return dict(bytes=byts, flops=flops)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(_device())


class _Dense:
    """H of a U(1) pivot on dense bonds: out = sum L[a] W[a, w] W[w, b] v R[b]."""

    def __init__(self, pd):
        self.pd = pd
        self.lo, self.nl = self._offsets(pd.left)
        self.ro, self.nr = self._offsets(pd.right)
        self.W = [_t(W.dense()) for W in (pd.W12, pd.W34) if W is not None]
        self.L = self._env(pd.L, pd.W12.aux_in, self.lo, self.nl)
        self.R = self._env(pd.R, (pd.W34 or pd.W12).aux_out, self.ro, self.nr)
        idx = np.empty(pd.vsize, dtype=np.int64)
        shape = (self.nl,) + tuple(w.shape[2] for w in self.W) + (self.nr,)
        for s, qin, qout, off, r, c in pd.block_offsets():
            at = tuple(pd.basis[s][1:]) if pd.nsite == 2 else (pd.basis[s][1],)
            i, j = np.meshgrid(self.lo[qin] + np.arange(r), self.ro[qout] + np.arange(c), indexing="ij")
            idx[off:off + r * c] = np.ravel_multi_index((i,) + at + (j,), shape).ravel(order="F")
        self.shape, self.idx = shape, _t(idx)

    @staticmethod
    def _offsets(sectors):
        off, o = {}, 0
        for q, d in sectors:
            off[tuple(q)] = o
            o += d
        return off, o

    def _env(self, sectors, aux, off, n):
        if isinstance(sectors, torch.Tensor):
            return sectors
        ao, na = self._offsets(aux)
        E = np.zeros((na, n, n))
        for qin, qout, qmid, blocks in sectors:
            for a, x in enumerate(blocks):
                E[ao[qmid] + a, off[qin]:off[qin] + x.shape[0], off[qout]:off[qout] + x.shape[1]] = x
        return _t(E)

    def __call__(self, v):
        x = torch.zeros(math.prod(self.shape), dtype=torch.float64, device=v.device)
        x[self.idx] = v
        x = x.reshape(self.nl, -1)
        T = torch.stack([La @ x for La in self.L])              # [a, x, rest]
        inner = self.shape[1:-1]
        for n, W in enumerate(self.W):                          # [a, x, (s'..), s, (rest)] -> [b, x, (s'..s'), rest]
            pre = math.prod(inner[:n])
            T = T.reshape(T.shape[0], self.nl * pre, inner[n], -1)
            out = torch.zeros((W.shape[1],) + tuple(T.shape[1:]), dtype=torch.float64, device=v.device)
            for a, b, p, q in torch.nonzero(W).tolist():
                out[b, :, p] += W[a, b, p, q] * T[a, :, q]
            T = out
        T = T.reshape(T.shape[0], -1, self.nr)
        y = torch.zeros_like(T[0])
        for Tb, Rb in zip(T, self.R):
            y += Tb @ Rb
        return y.reshape(-1)[self.idx]


def _blockwise(pd, vin):
    """H v of a pivot with SU(2) components, block by block."""
    L = {(qi, qo, qm, a): x for qi, qo, qm, bl in pd.L for a, x in enumerate(bl)}
    R = {(qi, qo, qm, a): x for qi, qo, qm, bl in pd.R for a, x in enumerate(bl)}
    place = {(s, qi, qo): (off, r, c) for s, qi, qo, off, r, c in pd.block_offsets()}
    v = _t(vin)

    def block(x, key):
        off, r, c = place[key]
        return x[off:off + r * c].reshape(c, r).T

    T, by_out, dev = {}, {}, ({}, {})
    for o, l, i, r, c in _terms(pd):
        d = by_out.setdefault((o, r), {})
        d[(l, i)] = d.get((l, i), 0.0) + c
    out = torch.zeros_like(v)
    for (o, r), terms in by_out.items():
        U = None
        for (l, i), c in terms.items():
            if (l, i) not in T:
                if l not in dev[0]:
                    dev[0][l] = _t(L[l])
                T[(l, i)] = dev[0][l] @ block(v, i)
            U = c * T[(l, i)] if U is None else U.add_(T[(l, i)], alpha=c)
        if r not in dev[1]:
            dev[1][r] = _t(R[r])
        block(out, o).add_(U @ dev[1][r])
    return out


def _lowest(H, v0):
    """Lowest eigenpair by Lanczos with full re-orthogonalisation; the vector's
    overlap with the start is positive, as a Ritz vector's is here."""
    Q, alpha, beta = [v0 / v0.norm()], [], []
    for k in range(300):
        w = H(Q[k])
        alpha.append(float(Q[k] @ w))
        B = torch.stack(Q)
        for _ in range(2):
            w = w - B.T @ (B @ w)
        beta.append(float(w.norm()))
        E, Y = np.linalg.eigh(np.diag(alpha) + np.diag(beta[:-1], 1) + np.diag(beta[:-1], -1))
        if beta[-1] * abs(Y[-1, 0]) < 1e-12 * max(1.0, abs(E[0])):
            break
        Q.append(w / beta[-1])
    psi = torch.stack(Q[:len(alpha)]).T @ _t(Y[:, 0])
    psi = psi / psi.norm()
    return float(E[0]), psi if float(psi @ v0) > 0 else -psi


def exact(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "advance":
        W, left, old, A, pd = _advance(case, rng)
        v = _vector([pd], rng)
        lo, nl = _Dense._offsets(left)
        mo, nm = _Dense._offsets(pd.left)
        X = _t(np.zeros((len(A), nl, nm)))
        for s, blocks in enumerate(A):
            for qin, qout, x in blocks:
                X[s, lo[qin]:lo[qin] + x.shape[0], mo[qout]:mo[qout] + x.shape[1]] = _t(x)
        Lold = _Dense._env(_Dense, old, W.aux_in, lo, nl)
        D = _t(W.dense())
        new = torch.zeros((D.shape[1], nm, nm), dtype=torch.float64, device=X.device)
        for a, b, p, q in torch.nonzero(D).tolist():
            new[b] += D[a, b, p, q] * (X[p].T.contiguous() @ (Lold[a] @ X[q]))
        pd.L = new
        return _Dense(pd)(_t(v))
    pds = _pivots(case, rng)
    v = _vector(pds, rng)
    energies, parts, off = [], [], 0
    for pd in pds:
        x = v[off:off + pd.vsize]
        off += pd.vsize
        if case["kind"] == "hxv":
            parts.append(_blockwise(pd, x) if pd.sym.non_abelian else _Dense(pd)(_t(x)))
        else:
            E, psi = _lowest(_Dense(pd), _t(x))
            energies.append(E)
            parts.append(psi)
    out = torch.cat(parts)
    if case["kind"] == "hxv":
        return out
    if case["kind"] == "lanczos":
        return dict(energy=energies[0], vector=out)
    return dict(energies=np.array(energies), vector=out)
