"""The two-lanes-per-block encoders and the four-per-thread decoder against the oracle, byte for byte: part-filled
workgroups (one block, one short of and one past a workgroup's 128), values at the midpoints of the code
tables and one unit to either side, signed zeros, subnormal and huge scales, NaN and infinities. The snap (decode of
encode) of blocks with NaN and infinities likewise, by rows, by columns and in a plan."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = ("Q8_0", "Q4_0", "F16", "Fp8E4M3", "Fp8E5M2", "Fp4")


@pytest.fixture(scope="module")
def fh():
    import ferrum_hip

    return ferrum_hip


@pytest.fixture(scope="module")
def g(fh):
    gpu = fh.Gpu.open_for_test()
    if gpu is None:
        pytest.skip("no gfx950 device")
    yield gpu
    gpu.close()


def blocks(nblocks, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((nblocks, 32)).astype(np.float32)
    # a quarter of the blocks: midpoints of the code tables (eighths, for a block maximum that makes the scale a
    # power of two), and their neighbours
    grid = rng.integers(-96, 97, (nblocks, 32)).astype(np.float32) / np.float32(8)
    grid[:, 0] = rng.choice(np.float32([12, 448, 57344, 127, 8, 7.999999]), nblocks)
    step = rng.integers(-1, 2, (nblocks, 32))
    grid = np.where(step < 0, np.nextafter(grid, np.float32(-np.inf)),
                    np.where(step > 0, np.nextafter(grid, np.float32(np.inf)), grid)).astype(np.float32)
    x = np.where((np.arange(nblocks) % 4 == 1)[:, None], grid, x)
    x *= np.exp2(rng.integers(-6, 7, nblocks)).astype(np.float32)[:, None]
    wide = np.arange(nblocks) % 8 == 2  # from subnormal to the largest floats
    x[wide] *= np.exp2(rng.integers(-140, 120, wide.sum()).astype(np.float64)).astype(np.float32)[:, None]
    x[rng.random(x.shape) < 0.05] = np.float32(-0.0)
    x[np.arange(nblocks) % 8 == 6] *= np.float32(0)
    return x


@pytest.mark.parametrize("kind", KINDS)
def test_encode_and_decode_at_the_edges(fh, g, orc, kind):
    kind = getattr(fh.QKind, kind)
    for nblocks in (1, 2, 127, 128, 129, 1031):
        x = blocks(nblocks, nblocks).reshape(-1)
        want = orc.encode(int(kind), x)
        packed = fh.encode(g, kind, g.upload(x), x.size)
        got = g.read_bytes(packed)[: want.size]
        assert np.array_equal(got, want), (kind, nblocks, np.flatnonzero(got != want)[:8])
        back = orc.decode(int(kind), want, x.size)
        dev = g.read(fh.decode(g, kind, packed, x.size))[: x.size]
        nan = np.isnan(back)
        assert np.array_equal(np.isnan(dev), nan)
        assert np.array_equal(dev[~nan].view(np.uint32), back[~nan].view(np.uint32)), (kind, nblocks)


@pytest.mark.parametrize("kind", ("Fp8E4M3", "Fp8E5M2", "Fp4"))
def test_encode_of_nan_and_infinity(fh, g, orc, kind):
    kind = getattr(fh.QKind, kind)
    x = blocks(160, 3)
    x[5, 3], x[5, 19], x[140, 31] = np.nan, -np.nan, np.nan
    x[9, 0], x[77, 16], x[78, 1] = np.inf, -np.inf, -np.inf
    x[78, 2] = np.nan
    x[79] = np.nan
    want = orc.encode(int(kind), x.reshape(-1))
    got = g.read_bytes(fh.encode(g, kind, g.upload(x.reshape(-1)), x.size))[: want.size]
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:8] // (want.size // 160)


def nonfinite():
    """160 blocks: all NaN, NaN in some lanes' or one lane's values only, infinities, both, and finite ones between."""
    x = blocks(160, 11)
    x[0], x[63], x[127], x[128], x[159] = np.nan, -np.nan, np.nan, np.nan, np.nan
    x[2, :4], x[3, 4:], x[64, ::2], x[65, 31], x[66, :16], x[67, 16:] = (np.nan,) * 6
    x[9, 0], x[77, 16], x[78, 1] = np.inf, -np.inf, -np.inf
    x[78, 2], x[79, 3] = np.nan, np.inf
    x[79, 4:] = np.nan
    return x


def same(got, want, what):
    """The bits of every value that is not NaN, and NaN where it is."""
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan), (what, np.flatnonzero(np.isnan(got) != nan)[:8])
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32)), what


@pytest.mark.parametrize("kind", ("Q8_0", "Q4_0"))
def test_encode_of_nan_and_infinity_q8_0_q4_0(fh, g, orc, kind):
    kind = getattr(fh.QKind, kind)
    x = nonfinite().reshape(-1)
    want = orc.encode(int(kind), x)
    got = g.read_bytes(fh.encode(g, kind, g.upload(x), x.size))[: want.size]
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:8] // (want.size // 160)


def test_snap_of_nan_and_infinity(fh, g, orc):
    x = nonfinite()
    rows = x.reshape(-1)
    cols = np.ascontiguousarray(x.T)  # a block down each of the 160 columns
    src, csrc = g.upload(rows), g.upload(cols.reshape(-1))
    want = orc.snap_rows(rows, 32)
    dst, cdst = g.zeros(rows.size), g.zeros(rows.size)
    fh.q8_snap_rows(g, src, dst, 32)
    same(g.read(dst), want, "rows")
    cwant = np.ascontiguousarray(want.reshape(160, 32).T).reshape(-1)
    fh.q8_snap_cols(g, csrc, cdst, (32, 160))
    same(g.read(cdst), cwant, "cols")
    pdst, pcdst = g.zeros(rows.size), g.zeros(rows.size)
    plan = fh.SnapPlan(g, [(fh.SNAP_ROWS, src, pdst, 32), (fh.SNAP_COLS, csrc, pcdst, (32, 160))])
    plan.run()
    same(g.read(pdst), want, "plan, rows")
    same(g.read(pcdst), cwant, "plan, cols")


def test_mxfp4_encode_of_the_largest_floats(fh, g, orc):
    """A block maximum within a few units of the largest float rounds to the next power of two in f32's log2: the codes
    for 8 and 12 then decode to infinity, and the nearest code is the one for 6. Maxima at the largest float, at and
    around the unit where the logarithm rounds up, at the start of the top binade and below it; the other values from
    tiny to the maximum, those past 7/8 of it and the code midpoints among them."""
    tops = np.uint32([0x7f7fffff, 0x7f7ffffe, 0x7f7fffd4, 0x7f7fffd3, 0x7f7fffd2, 0x7f7fff01, 0x7f7fff00, 0x7f7ffeff,
                      0x7f600000, 0x7f000000, 0x7effffff, 0x7effffd4]).view(np.float32)
    rng = np.random.default_rng(8)
    share = np.concatenate([rng.uniform(-1, 1, 19), [1, -1, 0.95, -0.95, 0.875, 0.8750001, 0.75, 0.625, 0.5, 0.4375, 1e-3,
                                                     1e-30, -0.0]]).astype(np.float32)
    x = np.concatenate([np.roll(share, s)[None] * t for t in tops for s in (0, 7)]).reshape(-1).astype(np.float32)
    assert np.isfinite(x).all()
    want = orc.encode(int(fh.QKind.Fp4), x)
    got = g.read_bytes(fh.encode(g, fh.QKind.Fp4, g.upload(x), x.size))[: want.size]
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:8] // 17
