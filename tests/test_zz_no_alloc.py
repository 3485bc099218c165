"""fh_linear_q_noalloc (no counterpart in the reference): the product without any device
allocation, its scratch taken from the library's static per-GPU array. Called through the C ABI,
its output must equal fh_linear_q_ptr's bit for bit (the same kernels on the same inputs), on two
calls in a row of which the second is smaller (the array keeps the first call's contents), for
every kernel path; and both stay within the reference's 1e-5 of the CPU product
(ferrum_wgpu/src/tolerance.rs:7) where the path keeps it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REDUCING = 1e-5


def say(*a):
    print(*a, flush=True)


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


def case(fh, g, orc, kind, rows, k, n, seed, cpu=True):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal(k * n) * 0.02).astype(np.float32)
    x = rng.standard_normal(rows * k).astype(np.float32)
    b = orc.quantise_matrix(int(kind), w, k, n)
    qw = fh.upload_qweight(g, kind, b, k, n)
    want = orc.matmul_tuned(x, orc.dequantised_in_out(int(kind), b, k, n), rows, k, n, 8) if cpu else None
    return qw, g.upload(x), g.zeros(rows * n), g.zeros(rows * n), want


# (path, rows, k, n): a larger product, then a smaller one, per path
PATHS = [
    ("Gemv", [(1, 4864, 896), (1, 896, 1152)]),
    ("Auto", [(1, 2048, 5632), (1, 768, 2304)]),
    ("Tiled", [(64, 2048, 2048), (8, 896, 1152)]),
    ("Auto", [(512, 896, 1152), (64, 896, 896)]),
    ("TiledF16", [(256, 2048, 2048), (32, 896, 1152)]),
    ("TiledFast", [(128, 896, 4864), (96, 896, 1152)]),
    ("Naive", [(4, 256, 320), (2, 64, 96)]),
]


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("path_name,shapes", PATHS, ids=[f"{p}-{s[0][0]}" for p, s in PATHS])
def test_noalloc_equals_linear_q_on_two_calls_in_a_row(fh, g, orc, kind_name, path_name, shapes):
    kind, path = fh.QKind[kind_name], fh.QPath[path_name]
    cases = [case(fh, g, orc, kind, r, k, n, 40 + i) for i, (r, k, n) in enumerate(shapes)]
    if path == fh.QPath.TiledFast:
        for qw, gx, ya, _, _ in cases:  # an ordinary fast product builds the correction operand
            fh.linear_q_with(g, gx, qw, ya, len(gx) // qw.k(), path)
    for (r, k, n), (qw, gx, ya, _, _) in zip(shapes, cases):
        fh.linear_q_ptr(g, gx.device_ptr(), qw, ya.device_ptr(), r, path)
    for (r, k, n), (qw, gx, _, yb, _) in zip(shapes, cases):
        say(f"noalloc {kind_name} {path_name} rows {r} {k}x{n}")
        fh.linear_q_noalloc(g, gx.device_ptr(), qw, yb.device_ptr(), r, path)
    for (r, k, n), (qw, gx, ya, yb, want) in zip(shapes, cases):
        a, b = g.read(ya), g.read(yb)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (path_name, r, k, n)
        e = orc.max_rel_err(b, want)
        say(f"  rows {r} {k}x{n}: bit-identical to linear_q, max rel err {e:.2e}")
        if path not in (fh.QPath.TiledFast, fh.QPath.TiledF16):
            assert e < REDUCING, (path_name, r, k, n, e)
        else:  # the MFMA-GEMM bound in the max norm
            assert np.abs(b - want).max() <= 1e-3 + 2e-3 * np.abs(want).max()


def test_noalloc_refuses_what_it_cannot_do_without_allocating(fh, g, orc):
    # more scratch than the array holds: the split x of 4096 rows of 4096 is 64 MiB
    qw, gx, ya, yb, _ = case(fh, g, orc, fh.QKind.Q4_0, 4096, 4096, 256, 7, cpu=False)
    with pytest.raises(fh.GpuError) as err:
        fh.linear_q_noalloc(g, gx.device_ptr(), qw, yb.device_ptr(), 4096, fh.QPath.Tiled)
    assert "scratch" in str(err.value)
    # the fast GEMM before its correction operand exists
    with pytest.raises(fh.GpuError) as err:
        fh.linear_q_noalloc(g, gx.device_ptr(), qw, yb.device_ptr(), 4096, fh.QPath.TiledFast)
    assert "correction operand" in str(err.value)
    with pytest.raises(fh.GpuError, match="null pointer"):
        fh._check(fh.lib().fh_linear_q_noalloc(g.handle, None, qw.handle, ctypes.c_void_p(yb.device_ptr()), 1, 0))
    # the device still works, and a product that fits runs
    fh.linear_q_noalloc(g, gx.device_ptr(), qw, yb.device_ptr(), 16, fh.QPath.Tiled)
    fh.linear_q_ptr(g, gx.device_ptr(), qw, ya.device_ptr(), 16, fh.QPath.Tiled)
    assert np.array_equal(g.read(ya)[:16 * 256], g.read(yb)[:16 * 256])


def test_noalloc_calls_through_two_handles_of_one_gpu_do_not_race(fh, g, orc):
    """Two handles of one GPU (two streams) share its one scratch array: each noalloc call waits
    for the previous one's work on that GPU, so interleaved calls through both handles, issued
    without any synchronisation between them, still equal linear_q_ptr's results bit for bit."""
    ordinal = int(__import__("os").environ.get("FERRUM_HIP_DEVICE", "0"))
    g2 = fh.Gpu(ordinal)
    work = []
    try:
        kind = fh.QKind.Q4_0
        for i, h in enumerate((g, g2, g, g2)):
            rows, k, n = (256, 2048, 2048) if i % 2 == 0 else (192, 2048, 1024)
            qw, gx, ya, yb, _ = case(fh, h, orc, kind, rows, k, n, 60 + i, cpu=False)
            fh.linear_q_ptr(h, gx.device_ptr(), qw, ya.device_ptr(), rows, fh.QPath.Tiled)
            work.append((h, qw, gx, ya, yb, rows))
        g.sync()
        g2.sync()
        for rep in range(3):
            for h, qw, gx, _, yb, rows in work:
                fh.linear_q_noalloc(h, gx.device_ptr(), qw, yb.device_ptr(), rows, fh.QPath.Tiled)
        g.sync()
        g2.sync()
        for i, (h, qw, gx, ya, yb, rows) in enumerate(work):
            assert np.array_equal(h.read(ya).view(np.uint32), h.read(yb).view(np.uint32)), i
        say("noalloc through two handles of one GPU: 12 interleaved calls equal linear_q_ptr")
    finally:
        for h, qw, gx, ya, yb, rows in work:
            for b in (gx, ya, yb):
                b.free()
            qw.free()
        g2.close()


def test_noalloc_refuses_overlapping_x_and_y(fh, g, orc):
    qw, gx, ya, yb, _ = case(fh, g, orc, fh.QKind.Q8_0, 8, 256, 256, 9, cpu=False)
    with pytest.raises(fh.GpuError, match="overlap"):
        fh.linear_q_noalloc(g, gx.device_ptr(), qw, gx.device_ptr() + 4 * 256, 8, fh.QPath.Rows)


# K-split one-launch products (eight splits each), then one with a single split
FEW = [(24, 4864, 896), (8, 5632, 1024), (5, 896, 300)]


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0", "Fp8E4M3", "Fp8E5M2", "Fp4", "F16"])
def test_noalloc_few_row_products_equal_linear_q(fh, g, orc, kind_name):
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(12)
    for rows, k, n in FEW + [(48, 896, 1152), (200, 1056, 257)]:
        raw = orc.encode(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32))
        qw, gx = fh.upload_qweight(g, kind, raw, k, n), g.upload(rng.standard_normal(rows * k).astype(np.float32))
        ya, yb = g.zeros(rows * n), g.zeros(rows * n)
        fh.linear_q_ptr(g, gx.device_ptr(), qw, ya.device_ptr(), rows)
        for _ in range(2):
            fh.linear_q_noalloc(g, gx.device_ptr(), qw, yb.device_ptr(), rows)
            assert np.array_equal(g.read(ya).view(np.uint32), g.read(yb).view(np.uint32)), (rows, k, n)


def test_captured_noalloc_products_beside_ordinary_ones(fh, g, orc):
    """A graph of no-allocation K-split products, replayed on a stream of its own while ordinary K-split products
    run on the handle's: neither touches the other's scratch or arrival counters, so both keep their bits."""
    hip = ctypes.CDLL("libamdhip64.so.7", mode=__import__("os").RTLD_NOLOAD | ctypes.RTLD_GLOBAL)
    P = ctypes.c_void_p

    def call(name, *a):
        assert getattr(hip, name)(*a) == 0, name

    work = []
    for kind_name in ("Q8_0", "Fp8E4M3"):
        for i, (rows, k, n) in enumerate(FEW):
            kind, rng = fh.QKind[kind_name], np.random.default_rng(30 + i)
            raw = orc.encode(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32))
            x = rng.standard_normal(rows * k).astype(np.float32)
            work.append((rows, fh.upload_qweight(g, kind, raw, k, n), g.upload(x), g.zeros(rows * n), g.zeros(rows * n)))
    for rows, qw, gx, ya, _ in work:
        fh.linear_q_ptr(g, gx.device_ptr(), qw, ya.device_ptr(), rows)
    want = [g.read(ya).copy() for *_, ya, _ in work]
    stream, graph, run = P(g.stream()), P(), P()
    call("hipStreamBeginCapture", stream, 2)  # relaxed
    for rows, qw, gx, _, yb in work:
        fh.linear_q_noalloc(g, gx.device_ptr(), qw, yb.device_ptr(), rows)
    call("hipStreamEndCapture", stream, ctypes.byref(graph))
    call("hipGraphInstantiate", ctypes.byref(run), graph, None, None, ctypes.c_size_t(0))
    other = P()
    call("hipStreamCreateWithFlags", ctypes.byref(other), 1)
    try:
        for rep in range(20):
            for _ in range(4):
                call("hipGraphLaunch", run, other)
            for _ in range(8):
                for rows, qw, gx, ya, _ in work:
                    fh.linear_q_ptr(g, gx.device_ptr(), qw, ya.device_ptr(), rows)
            call("hipStreamSynchronize", other)
            g.sync()
            for (rows, qw, gx, ya, yb), w in zip(work, want):
                assert np.array_equal(g.read(ya).view(np.uint32), w.view(np.uint32)), (rep, rows, "ordinary")
                assert np.array_equal(g.read(yb).view(np.uint32), w.view(np.uint32)), (rep, rows, "captured")
    finally:
        call("hipGraphExecDestroy", run)
        call("hipGraphDestroy", graph)
        call("hipStreamDestroy", other)


@pytest.mark.parametrize("kind_name,rows,k,n", [("Fp8E4M3", 2048, 896, 1152), ("Fp4", 1736, 640, 2474), ("F16", 1204, 5760, 1079),
                                                ("Q8_0", 2038, 2080, 10676)])
def test_noalloc_takes_products_whose_kernel_needs_more_scratch(fh, g, orc, kind_name, rows, k, n):
    """K splits whose partial sums do not fit the array: the ring kernel needs split x alone. Its sums are in another
    order: within the bound that any order keeps (test_gpu_ring_gemm.py)."""
    kind, rng = fh.QKind[kind_name], np.random.default_rng(k)
    raw = orc.encode(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32))
    w = orc.decode(int(kind), raw, k * n).reshape(n, k).T.astype(np.float64)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    qw, gx, gy = fh.upload_qweight(g, kind, raw, k, n), g.upload(x), g.zeros(rows * n)
    fh.linear_q_noalloc(g, gx.device_ptr(), qw, gy.device_ptr(), rows, fh.QPath.Tiled)
    first = g.read(gy).copy()
    fh.linear_q_noalloc(g, gx.device_ptr(), qw, gy.device_ptr(), rows, fh.QPath.Tiled)
    got = g.read(gy)
    assert np.array_equal(first.view(np.uint32), got.view(np.uint32))
    pick = np.r_[0:40, rows - 40:rows]
    err = np.abs(got.reshape(rows, n)[pick] - x[pick].astype(np.float64) @ w)
    assert np.all(err <= (k + 8) * 2.0**-24 * (np.abs(x[pick]).astype(np.float64) @ np.abs(w)))
    fh.linear_q_ptr(g, gx.device_ptr(), qw, gy.device_ptr(), rows, fh.QPath.Tiled)
    assert not np.array_equal(g.read(gy).view(np.uint32), got.view(np.uint32))  # (the kernel with K splits)
