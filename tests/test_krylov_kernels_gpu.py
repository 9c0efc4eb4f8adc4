"""The vector kernels of the eigensolvers at the sizes where they can go wrong:
the weighted dot product's segments, the Gram-Schmidt passes of long vectors and
long bases, the conjugate-gradient passes of the refinement, and a batch that
converges with its next iterations already queued."""
import ctypes
import math
import sys

import numpy as np
import pytest

from vmps_amd import _lib, models, synth
from vmps_amd.pivot import DeviceVector, HxV, PivotBatch, PivotMatrix2, dot, lanczos, lanczos_batch

sys.path.insert(0, __file__.rsplit("/", 1)[0])
import pivots  # noqa: E402

pytestmark = pytest.mark.gpu


def _weights(pd):
    return np.concatenate([np.full(r * c, pd.sym.coeff_dot(qo)) for (_, _, qo, _, r, c) in pd.block_offsets()])


def _chain(n, M, seed=3):
    W = models.heisenberg_u1_mpo()
    return synth.make_pivot(W, W, synth.heisenberg_bond(n, M), synth.heisenberg_bond(n + 2, M),
                            np.random.default_rng(seed), hermitian=True)


# ---- weighted dot product ------------------------------------------------------
def _check_dot(pd):
    H = PivotMatrix2(pd)
    w = _weights(pd)
    rng = np.random.default_rng(7)
    x, y = rng.standard_normal(pd.vsize), rng.standard_normal(pd.vsize)
    terms = w * x * y
    ref = math.fsum(terms)
    # a lane adds at most 64 products, then 6 + 3 additions in the workgroup, and the
    # second pass nseg / 1024 + 8: fewer than 100 roundings of 2^-53 in a chain
    tol = 100 * 2.0 ** -53 * np.abs(terms).sum()
    dx, dy = DeviceVector(H, x), DeviceVector(H, y)
    r = ctypes.c_double()
    _lib.check(H._lib.vmps_vec_dot(H._plan, dx.ptr, dy.ptr, ctypes.byref(r)))
    assert abs(r.value - ref) <= tol
    assert dot(H, x, y) == r.value
    dx.free()
    dy.free()


@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 9), (8, 8), (5, 13), (7, 73), (16, 32), (19, 27), (45, 91),
                                       (64, 64), (17, 241), (90, 91), (128, 96)])
def test_dot_segment_lengths(rows, cols):
    """Blocks of 1, 63 to 65, 511 to 513, 4095 to 4097, 8190 and 12288 elements:
    segments of at most 4096, a wave's 512 per round."""
    W = models.heisenberg_u1_mpo()
    print("dot of blocks of", rows * cols, flush=True)
    _check_dot(synth.make_pivot(W, W, [((-1,), rows), ((1,), 2)], [((-1,), cols), ((1,), 3)],
                                np.random.default_rng(rows)))


def test_dot_weights():
    """SU(2) blocks, weighted by their multiplets' dimensions."""
    W = models.heisenberg_su2_mpo()
    pd = synth.make_pivot(W, W, synth.heisenberg_su2_bond(10, 60), synth.heisenberg_su2_bond(12, 60),
                          np.random.default_rng(2))
    assert len(set(_weights(pd))) > 2
    _check_dot(pd)


# ---- Gram-Schmidt of long vectors and long bases -----------------------------------
def _host_lanczos(H, v0, iters):
    """Ritz values after each iteration of a fully re-orthogonalised numpy run on
    the plan's HxV (weights 1)."""
    Q = np.empty((iters + 1, v0.size))
    Q[0] = v0 / np.linalg.norm(v0)
    al, be, out = [], [], []
    for k in range(iters):
        x = HxV(H, Q[k])
        a = 0.0
        for _ in range(2):
            c = Q[:k + 1] @ x
            x -= c @ Q[:k + 1]
            a += c[k]
        al.append(a)
        T = np.diag(al) + np.diag(be, 1) + np.diag(be, -1)
        out.append(np.linalg.eigvalsh(T)[0])
        be.append(np.linalg.norm(x))
        Q[k + 1] = x / be[-1]
    return out


def _check_long(pd, H, counts):
    v0 = np.random.default_rng(4).uniform(-1, 1, pd.vsize)
    ref = _host_lanczos(H, v0, max(counts))
    for iters in counts:
        o = dict(v0=v0, max_iter=iters, tol_eigval=0.0, tol_state=0.0)
        vg, rg = lanczos(H, graph=True, **o)
        ve, re_ = lanczos(H, graph=False, **o)
        print("iterations", rg["iterations"], "energy", rg["energy"], "host", ref[iters - 1], flush=True)
        assert rg["iterations"] == iters
        # as for the other bases: the Ritz value of a semi-orthogonal basis to rounding
        assert abs(rg["energy"] - ref[iters - 1]) <= 1e-11 * abs(ref[iters - 1])
        assert rg["energy"] == re_["energy"] and np.array_equal(vg, ve)


@pytest.mark.parametrize("n,M", [(8, 40), (9, 60)])  # 1352 and 2880 elements, not multiples of 256
def test_long_basis_on_short_vectors(n, M):
    """A plan whose basis has room for more than 512 vectors forms the row sums in
    their own kernel; rows past the 36 that a workgroup keeps are read again."""
    pd = _chain(n, M)
    assert pd.vsize % 256
    H = PivotMatrix2(pd)
    print("long basis, vsize", pd.vsize, flush=True)
    _, r = lanczos(H, max_iter=600, tol_eigval=1e-12, tol_state=1e-9)  # the basis stays allocated
    assert r["converged"]
    _check_long(pd, H, (2, 16, 17, 35, 36, 37, 38, 53))


def test_long_vectors():
    """Vectors of more than 64 x 8192 elements."""
    pd = _chain(20, 990)
    assert pd.vsize > 64 * 8192 and pd.vsize % 256
    print("long vectors, vsize", pd.vsize, flush=True)
    _check_long(pd, PivotMatrix2(pd), (7, 36, 37, 50))


# ---- conjugate-gradient corrections ----------------------------------------------
def _residual(H64, v):
    hv = HxV(H64, v)
    e = v @ hv / (v @ v)
    return e, np.linalg.norm(hv - e * v) / np.linalg.norm(v), np.linalg.norm(hv)


@pytest.mark.parametrize("n,M", [(5, 10), (8, 40), (14, 520)])  # 116, 1352 and over 512 x 256 elements
@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
def test_corrections_reach_the_fp64_residual(n, M, prec):
    """The refined pair is an FP64 eigenpair to the tolerance asked for, and the one
    that the FP64 solve finds; energies and residuals are those of the vector."""
    pd = _chain(n, M)
    H64 = PivotMatrix2(pd)
    H = PivotMatrix2(pd, precision=prec)
    print("corrections", prec, "vsize", pd.vsize, flush=True)
    it = min(300, pd.vsize)
    v64, r64 = lanczos(H64, max_iter=it, tol_eigval=1e-13, tol_state=1e-9)
    v, r = lanczos(H, precision=prec, max_iter=it, tol_eigval=1e-6, tol_state=1e-3, refine_tol_eigval=1e-12,
                   refine_tol_state=1e-8)
    e, res, norm = _residual(H64, v)
    print(r, r64["energy"], e, res, flush=True)
    assert r["converged"] and r["refine_cg"] > 0
    assert abs(np.linalg.norm(v) - 1.0) <= 1e-12
    # Hv carried through the update against a new product: a few roundings of ||Hv||
    assert abs(e - r["energy"]) <= 1e-13 * max(1.0, norm) and abs(res - r["residual"]) <= 1e-12 * max(1.0, norm)
    assert res <= 1.001e-8
    # both are eigenvectors to 1e-8; their distance is that over the gap (some 1e-2)
    assert abs(r["energy"] - r64["energy"]) <= 1e-12 * max(1.0, abs(e))
    assert abs(abs(v @ v64) - 1.0) <= 1e-8


def test_corrections_on_an_indefinite_operator():
    """After one step from a random vector the Ritz value is above several
    eigenvalues: a direction of negative curvature ends the conjugate gradients,
    whose last correction is kept.  The FP64 Rayleigh-Ritz step cannot raise the
    energy; the result is repeatable."""
    pd = _chain(8, 40)
    H64 = PivotMatrix2(pd)
    H = PivotMatrix2(pd, precision="bf16x3")
    v0 = np.random.default_rng(5).uniform(-1, 1, pd.vsize)
    o = dict(v0=v0, precision="bf16x3", max_iter=2, tol_eigval=0.0, tol_state=0.0, refine_tol_eigval=1e-12,
             refine_tol_state=1e-9)
    v, r = lanczos(H, **o)
    e, res, norm = _residual(H64, v)
    print(r, e, res, flush=True)
    assert np.isfinite(v).all() and abs(np.linalg.norm(v) - 1.0) <= 1e-12
    # energy_mixed: the Rayleigh quotient of the vector that the corrections start from
    assert r["energy"] <= r["energy_mixed"] + 1e-12 * norm
    assert abs(e - r["energy"]) <= 1e-12 * max(1.0, norm)
    v2, r2 = lanczos(H, **o)
    assert np.array_equal(v, v2) and r2["refine_cg"] == r["refine_cg"]


# ---- a batch converging with iterations queued -------------------------------------
def test_batch_ends_with_iterations_queued():
    """Pivots of 24 to 46 elements: the residual estimate is far from its tolerance
    until the Krylov space ends, so the last iterations queued are not needed (the
    HxV count shows them).  The eigenpairs are those without them, bit for
    bit, and those of the dense matrices."""
    pds = [_chain(n, M, seed=n + M) for n, M in ((3, 4), (4, 4), (4, 6))]
    B = PivotBatch(pds)
    v0 = np.random.default_rng(6).uniform(-1, 1, B.vsize)
    o = dict(v0=v0, max_iter=120, tol_eigval=1e-13, tol_state=1e-11)
    vg, rg = lanczos_batch(B, graph=True, **o)
    ve, re_ = lanczos_batch(B, graph=False, **o)
    it = max(r["iterations"] for r in rg)
    print("iterations", [r["iterations"] for r in rg], "hxv", rg[0]["hxv_calls"], re_[0]["hxv_calls"], flush=True)
    assert rg[0]["hxv_calls"] == 4 * ((it + 3) // 4) + 4 + 1
    assert np.array_equal(vg, ve)
    for pd, r, re1, v in zip(pds, rg, re_, B.split(vg)):
        assert r["converged"] and r["energy"] == re1["energy"] and r["iterations"] == re1["iterations"]
        H = PivotMatrix2(pd)
        A = np.stack([HxV(H, x) for x in np.eye(pd.vsize)], axis=1)
        e, u = np.linalg.eigh(0.5 * (A + A.T))
        assert abs(r["energy"] - e[0]) <= 1e-12 * max(1.0, np.abs(e).max())
        if e[1] - e[0] > 1e-3 * np.abs(e).max():
            assert abs(abs(u[:, 0] @ v) - 1.0) <= 1e-10
