"""Tile configurations and the autotuner: every configuration gives the
oracle's HxV (FP64: 1e-12 relative; split-BF16 x3: 5e-5), the autotuner picks
one of its candidates and caches it per block-size histogram."""
import sys

import numpy as np
import pytest

import oracle
from vmps_amd import _lib, synth
from vmps_amd.pivot import DeviceVector, HxV, PivotMatrix2, clear_tile_cache

sys.path.insert(0, __file__.rsplit("/", 1)[0])
import pivots  # noqa: E402

pytestmark = pytest.mark.gpu

FP64_RTOL = 1e-12
BF16X3_RTOL = 5e-5


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.fixture(scope="module")
def case():
    # blocks up to ~150, so that the 128 x 128 split-BF16 tiles are used for some
    pd = pivots.small_heisenberg(seed=3, M=400, nleft=6)
    v = synth.random_vector(pd, 4)
    lib = oracle.load()
    h = pivots.build_oracle(lib, pd)
    try:
        ref = pivots.oracle_hxv(lib, h, v, nthreads=8)
    finally:
        lib.oracle_pivot2_destroy(h)
    return pd, v, ref


@pytest.mark.parametrize("edge", [16, 32])
def test_fp64_wave_edges(case, edge):
    pd, v, ref = case
    print("fp64 wave edge", edge, "vsize", pd.vsize, flush=True)
    H = PivotMatrix2(pd)
    H.set_tiles(edge, H.tiles()["big_min"])
    assert H.tiles()["wave_edge"] == edge
    assert _rel(HxV(H, v), ref) <= FP64_RTOL


@pytest.mark.parametrize("big_min", [96, 64, 0])
def test_bf16x3_big_thresholds(case, big_min):
    pd, v, ref = case
    print("bf16x3 big_min", big_min, flush=True)
    H = PivotMatrix2(pd, precision="bf16x3")
    H.set_tiles(H.tiles()["wave_edge"], big_min)
    assert H.tiles()["big_min"] == big_min
    assert _rel(HxV(H, v), ref) <= BF16X3_RTOL


@pytest.mark.parametrize("precision,tol", [("fp64", FP64_RTOL), ("fp32", 1e-5), ("bf16x3", BF16X3_RTOL)])
@pytest.mark.parametrize("which", ["heis", "lr40"])
def test_explicit_stage_b(case, precision, tol, which):
    """U = sum c T formed by its own kernel, stage C reading U: same result as
    the fused combine (and the oracle), on the D_W = 5 chain and on the
    long-range D_W = 40 SU(2) pivot with many terms per output block."""
    if which == "heis":
        pd, v, ref = case
    else:
        pd = synth.make_workload("heisenberg_su2_lr40_L60_M1024", M=96)
        v = synth.random_vector(pd, 8)
        lib = oracle.load()
        h = pivots.build_oracle(lib, pd)
        try:
            ref = pivots.oracle_hxv(lib, h, v, nthreads=8)
        finally:
            lib.oracle_pivot2_destroy(h)
    print("explicit stage B", which, precision, flush=True)
    H = PivotMatrix2(pd, precision=precision)
    fused = HxV(H, v)
    H.set_tiles(explicit_u=1)
    assert H.tiles()["explicit_u"] == 1
    out = HxV(H, v)
    assert _rel(out, ref) <= tol
    assert _rel(out, fused) <= (1e-15 if precision == "fp64" else 2 * tol)
    H.set_tiles(explicit_u=0)  # and back
    assert _rel(HxV(H, v), fused) == 0.0


@pytest.mark.parametrize("precision,tol", [("fp64", FP64_RTOL), ("fp32", 1e-5), ("bf16x3", BF16X3_RTOL)])
def test_autotune_picks_candidate_and_caches(case, precision, tol):
    pd, v, ref = case
    print("autotune", precision, flush=True)
    H = PivotMatrix2(pd, precision=precision)
    cfg = H.autotune(iters=3)
    if cfg["from_cache"] == 0:
        assert cfg["n_tried"] >= 2 and cfg["ms"] > 0
    if precision == "bf16x3":
        assert cfg["big_min"] in (96, 192, 0)
    else:
        assert cfg["wave_edge"] in (16, 32)
    assert _rel(HxV(H, v), ref) <= tol
    # a second plan of the same shape takes the cached choice without timing
    H2 = PivotMatrix2(pd, precision=precision)
    cfg2 = H2.autotune(iters=3)
    assert cfg2["from_cache"] == 1
    assert (cfg2["wave_edge"], cfg2["big_min"], cfg2["explicit_u"]) == (cfg["wave_edge"], cfg["big_min"],
                                                                      cfg["explicit_u"])
    assert _rel(HxV(H2, v), ref) <= tol
    # after the cache is cleared, the next plan of that shape is timed again
    clear_tile_cache()
    H3 = PivotMatrix2(pd, precision=precision)
    cfg3 = H3.autotune(iters=3)
    assert cfg3["from_cache"] == 0 and cfg3["n_tried"] >= 2
    assert _rel(HxV(H3, v), ref) <= tol


def test_set_tiles_rejects_bad_edge(case):
    pd, _, _ = case
    H = PivotMatrix2(pd)
    with pytest.raises(Exception):
        H.set_tiles(24, 96)


@pytest.mark.parametrize("precision,tol", [("fp64", FP64_RTOL), ("fp32", 1e-5)])
@pytest.mark.parametrize("big_min64,xu", [(96, 0), (64, 1), (128, 1)])
def test_fp64_fp32_big_tiles(case, precision, tol, big_min64, xu):
    """LDS-staged FP64 / FP32 tiles, 64 wide on a pivot of this size, for the
    problems >= big_min64 (with the fused and with the explicit stage B) against the
    oracle; FP64 is bit-identical to the wave tiles only up to summation order."""
    pd, v, ref = case
    print("big tiles", precision, big_min64, xu, flush=True)
    H = PivotMatrix2(pd, precision=precision)
    H.set_tiles(big_min64=big_min64, explicit_u=xu)
    cfg = H.tiles()
    assert cfg["big_min64"] == big_min64 and cfg["explicit_u"] == xu
    assert _rel(HxV(H, v), ref) <= tol


# sector dimensions at the edges of the 16 x 16 accumulators, 32-row steps, 16-deep K
# steps and 64-wide tiles of the LDS-staged kernels, odd ones among them
EDGE_LEFT = [((-5,), 1), ((-3,), 17), ((-1,), 64), ((1,), 65), ((3,), 33), ((5,), 130), ((7,), 2)]
EDGE_RIGHT = [((-5,), 3), ((-3,), 16), ((-1,), 127), ((1,), 31), ((3,), 96), ((5,), 48), ((7,), 15)]


@pytest.fixture(scope="module")
def edge_case():
    from vmps_amd import models
    W = models.heisenberg_u1_mpo()
    pd = synth.make_pivot(W, W, EDGE_LEFT, EDGE_RIGHT, np.random.default_rng(12))
    v = synth.random_vector(pd, 13)
    lib = oracle.load()
    h = pivots.build_oracle(lib, pd)
    try:
        return pd, v, pivots.oracle_hxv(lib, h, v, nthreads=8)
    finally:
        lib.oracle_pivot2_destroy(h)


@pytest.mark.parametrize("precision,tol", [("fp64", FP64_RTOL), ("fp32", 1e-5)])
@pytest.mark.parametrize("big_min64,xu", [(1, 1), (1, 0), (33, 1)])
def test_lds_tiles_at_block_edges(edge_case, precision, tol, big_min64, xu):
    pd, v, ref = edge_case
    print("LDS tiles at edges", precision, big_min64, xu, flush=True)
    H = PivotMatrix2(pd, precision=precision)
    H.set_tiles(big_min64=big_min64, explicit_u=xu)
    assert _rel(HxV(H, v), ref) <= tol


@pytest.mark.parametrize("precision,tol", [("fp64", FP64_RTOL), ("fp32", 1e-5)])
@pytest.mark.parametrize("edge", [16, 32])
def test_wave_tiles_at_block_edges(edge_case, precision, tol, edge):
    pd, v, ref = edge_case
    print("wave tiles at edges", precision, edge, flush=True)
    H = PivotMatrix2(pd, precision=precision)
    H.set_tiles(wave_edge=edge, big_min64=0, explicit_u=0)
    assert _rel(HxV(H, v), ref) <= tol


@pytest.mark.parametrize("big_min,xu", [(1, 1), (1, 0), (33, 1), (0, 1)])
def test_bf16x3_tiles_at_block_edges(edge_case, big_min, xu):
    pd, v, ref = edge_case
    print("split-BF16 tiles at edges", big_min, xu, flush=True)
    H = PivotMatrix2(pd, precision="bf16x3")
    H.set_tiles(big_min=big_min, explicit_u=xu)
    assert _rel(HxV(H, v), ref) <= BF16X3_RTOL


def _tiles128(pd):
    """128 x 128 tiles of the vector's blocks of 128 and more.  From 256 on the FP64
    and FP32 LDS tiles are 128 wide instead of 64, and split-BF16 stage C's 128 x 256
    with the explicit stage B (the rule itself: tests/plan/plan_check.cpp)."""
    return sum(-(-r // 128) * -(-c // 128) for (_, _, _, _, r, c) in pd.block_offsets() if min(r, c) >= 128)


@pytest.mark.parametrize("M,nleft", [(640, 29), (2047, 30)])
def test_lds_tiles_split_k(M, nleft):
    """Stage C tiles cut along K, FP64 in 64-wide tiles and split-BF16 in 128 x 128
    ones, against the wave tiles: both sum a few thousand products per element
    in FP64, so they agree to 1e-13 of the result's norm.  The split-BF16 tiles
    against that result."""
    from vmps_amd import models
    W = models.heisenberg_su2_lr_mpo(synth.lr_couplings(3, np.random.default_rng(1)))
    pd = synth.make_pivot(W, W, synth.heisenberg_su2_bond(nleft, M), synth.heisenberg_su2_bond(nleft + 2, M),
                          np.random.default_rng(14))
    v = synth.random_vector(pd, 15)
    print("split K", M, "vsize", pd.vsize, flush=True)
    assert _tiles128(pd) < 256
    H = PivotMatrix2(pd)
    H.set_tiles(big_min64=0, explicit_u=0)
    ref = HxV(H, v)
    H.set_tiles(big_min64=1, explicit_u=1)
    out = HxV(H, v)
    assert _rel(out, ref) <= 1e-13
    assert np.array_equal(HxV(H, v), out)  # a fixed order of summation
    H.set_precision("bf16x3")
    H.set_tiles(big_min=1, explicit_u=1)
    out = HxV(H, v)
    assert _rel(out, ref) <= BF16X3_RTOL
    assert np.array_equal(HxV(H, v), out)


@pytest.fixture(scope="module")
def wide_case():
    """A pivot of over 256 128 x 128 tiles, the last of each block 1 to 4 strips of 32
    rows and 32 or 64 columns wide, and its HxV on the FP64 wave tiles."""
    from vmps_amd import models
    W = models.heisenberg_u1_mpo()
    left = [((-1,), 641), ((1,), 700), ((3,), 736), ((5,), 765)]
    right = [((-1,), 769), ((1,), 595), ((3,), 935), ((5,), 1020)]
    pd = synth.make_pivot(W, W, left, right, np.random.default_rng(21))
    v = synth.random_vector(pd, 22)
    assert _tiles128(pd) >= 256
    H = PivotMatrix2(pd)
    H.set_tiles(wave_edge=32, big_min64=0, explicit_u=0)
    return pd, v, HxV(H, v)


@pytest.mark.parametrize("xu", [1, 0])
def test_bf16x3_wide_tiles_at_block_edges(wide_case, xu):
    """Stage C's split-BF16 tiles of such a pivot: 128 x 256 with the explicit stage B,
    128 x 128 with the fused one, against the FP64 wave tiles."""
    pd, v, ref = wide_case
    print("wide split-BF16 tiles, vsize", pd.vsize, xu, flush=True)
    H = PivotMatrix2(pd, precision="bf16x3")
    H.set_tiles(big_min=1, explicit_u=xu)
    out = HxV(H, v)
    assert _rel(out, ref) <= BF16X3_RTOL
    assert np.array_equal(HxV(H, v), out)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 1e-5)])
@pytest.mark.parametrize("xu", [1, 0])
def test_128_wide_tiles_at_block_edges(wide_case, precision, tol, xu):
    """The 128-wide FP64 and FP32 tiles, stage B explicit and fused, against the FP64
    wave tiles (a few thousand products per element on both sides)."""
    pd, v, ref = wide_case
    print("128-wide tiles, vsize", pd.vsize, precision, xu, flush=True)
    H = PivotMatrix2(pd, precision=precision)
    H.set_tiles(big_min64=1, explicit_u=xu)
    out = HxV(H, v)
    assert _rel(out, ref) <= tol
    assert np.array_equal(HxV(H, v), out)


@pytest.mark.parametrize("precision,tol", [("fp64", FP64_RTOL), ("bf16x3", BF16X3_RTOL)])
def test_large_sectors_with_thin_blocks(precision, tol):
    """A sector of 260 and more does not put every problem on the LDS-staged
    tiles while the blocks are thin; the tuner's choice gives the same HxV."""
    from vmps_amd import models
    W = models.heisenberg_u1_mpo()
    pd = synth.make_pivot(W, W, [((-1,), 260), ((1,), 5), ((3,), 40)], [((-1,), 3), ((1,), 4), ((3,), 30)],
                          np.random.default_rng(23))
    v = synth.random_vector(pd, 24)
    print("thin blocks", precision, "vsize", pd.vsize, flush=True)
    lib = oracle.load()
    h = pivots.build_oracle(lib, pd)
    try:
        ref = pivots.oracle_hxv(lib, h, v, nthreads=8)
    finally:
        lib.oracle_pivot2_destroy(h)
    H = PivotMatrix2(pd, precision=precision)
    cfg = H.tiles()
    assert cfg["big_min64"] == 128 and cfg["big_min"] == 96 and cfg["explicit_u"] == 1
    assert _rel(HxV(H, v), ref) <= tol
    H.autotune(iters=2)
    assert _rel(HxV(H, v), ref) <= tol


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("tiles", [dict(wave_edge=16, big_min64=0, big_min=0, explicit_u=0),
                                   dict(wave_edge=32, big_min64=0, big_min=0, explicit_u=1),
                                   dict(big_min64=1, big_min=1, explicit_u=0),
                                   dict(big_min64=1, big_min=1, explicit_u=1)])
def test_nan_stays_in_its_blocks(edge_case, precision, tiles):
    """A vector block of NaN reaches the outputs its terms lead to and no other:
    an operand's elements past K are zeros, not the memory behind the block (a
    zero of the other operand would hide finite memory, not NaN).  The other
    outputs keep every bit; which ones they are, the FP64 product of the block
    alone says."""
    pd, v, _ = edge_case
    print("NaN blocks", precision, tiles, flush=True)
    probe = PivotMatrix2(pd)
    H = PivotMatrix2(pd, precision=precision)
    H.set_tiles(**tiles)
    din, dout = DeviceVector(H, v), DeviceVector(H)

    def apply(x):
        din.upload(x)
        _lib.check(H._lib.vmps_hxv_device(H._plan, din.ptr, dout.ptr, None))
        return dout.download()

    clean = apply(v)
    checked = 0
    for (_, _, _, off, rows, cols) in pd.block_offsets():
        sl = slice(off, off + rows * cols)
        alone = np.zeros_like(v)
        alone[sl] = v[sl]
        free = HxV(probe, alone) == 0.0
        x = v.copy()
        x[sl] = np.nan
        out = apply(x)
        assert np.array_equal(out[free], clean[free])
        assert np.isnan(out).any()
        checked += int(free.any())
    assert checked > 10
    din.free()
    dout.free()


def _large_pivot():
    from vmps_amd import models
    W = models.heisenberg_u1_mpo()
    return synth.make_pivot(W, W, [((-1,), 300), ((1,), 280)], [((-1,), 290), ((1,), 257)], np.random.default_rng(41))


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
def test_autotune_of_a_large_pivot_drops_hand_set_tiles(precision):
    """A pivot dominated by large blocks is tuned among its rule's own choices: a
    slow configuration set by hand before is neither kept nor cached, and the
    other precisions' threshold does not travel with the choice."""
    pd = _large_pivot()
    print("hand-set tiles, then autotune", precision, flush=True)
    clear_tile_cache()
    H = PivotMatrix2(pd, precision=precision)
    assert H.tiles()["big_min"] == 1 and H.tiles()["big_min64"] == 1
    H.set_tiles(big_min=512, big_min64=512, explicit_u=0)
    cfg = H.autotune(iters=1)
    used = "big_min" if precision == "bf16x3" else "big_min64"
    assert cfg[used] in (0, 1) and cfg["explicit_u"] == 1
    H2 = PivotMatrix2(pd, precision=precision)
    cfg2 = H2.autotune(iters=1)
    assert cfg2["from_cache"] == 1 and cfg2[used] == cfg[used] and cfg2["explicit_u"] == 1
    assert cfg2["big_min64" if precision == "bf16x3" else "big_min"] == 1
