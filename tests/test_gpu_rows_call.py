"""AUTO's one-launch few-row product (2 to 64 rows, one linear_q per product) against the float64
product of the stored weights, every output held to the summation error bound of any order (as
test_gpu_rows.py: (k + 8) 2^-24 sum_k |x_k w_k|).

Sizes: one and two 32-row tiles and their edges; block counts below a wavefront's pair, odd, not a
multiple of the eight wavefronts' pairs, and deep enough to split K over workgroups (with a remainder);
outputs that are not whole tiles, one and two tiles per workgroup (257 to 512 tiles: an odd count, whose
last workgroup has one tile, with a last tile of 5 outputs), and a count past that, which the other few-row kernels take;
x at a 4-byte offset. Each product runs twice with another between them: the K splits' tickets must be left at zero
and the sums must not depend on which workgroup ends last."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("k,n", [(32, 1), (96, 33), (544, 300), (1056, 40), (4864, 100), (3104, 257), (64, 16450),
                                 (64, 8261), (544, 8197), (896, 11237)])
def test_one_launch_product(fh, g, orc, kind_name, k, n):
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(k + n)
    b = orc.quantise_matrix(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32), k, n)
    w = orc.dequantised_in_out(int(kind), b, k, n).reshape(k, n).astype(np.float64)
    qw = fh.upload_qweight(g, kind, b, k, n)
    for m in (2, 3, 31, 32, 33, 64):
        x = rng.standard_normal((m, k)).astype(np.float32)
        gx, gy = g.upload(np.concatenate([[0.0], x.reshape(-1)])), g.zeros(m * n)
        other = g.zeros(m * n)
        fh.linear_q_ptr(g, gx.device_ptr() + 4, qw, gy.device_ptr(), m)
        first = g.read(gy)
        fh.linear_q_ptr(g, gx.device_ptr(), qw, other.device_ptr(), m)
        fh.linear_q_ptr(g, gx.device_ptr() + 4, qw, gy.device_ptr(), m)
        got = g.read(gy)
        assert np.array_equal(first.view(np.uint32), got.view(np.uint32)), (kind_name, k, n, m)
        bound = (k + 8) * 2.0**-24 * (np.abs(x).astype(np.float64) @ np.abs(w))
        err = np.abs(got.reshape(m, n) - x.astype(np.float64) @ w)
        assert np.all(err <= bound), (kind_name, k, n, m, float((err / np.maximum(bound, 1e-38)).max()))
        print(f"{kind_name} {k}x{n} rows {m}: {float((err / np.maximum(bound, 1e-38)).max()):.3f} of the bound", flush=True)


@pytest.mark.parametrize("kind_name", ["Fp8E4M3", "Fp8E5M2", "Fp4", "F16"])
@pytest.mark.parametrize("k,n", [(32, 1), (96, 33), (1056, 40), (4864, 100), (64, 16450), (64, 8261), (544, 8197),
                                 (896, 11237)])
def test_one_launch_product_of_gguf_rows(fh, g, orc, kind_name, k, n):
    """The formats kept as GGUF rows. In the first output's last block and the last output's first one an
    infinity or NaN makes that output NaN for every row of x, and no other."""
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(k + n)
    raw = orc.encode(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32))
    w = orc.decode(int(kind), raw, k * n).reshape(n, k).T.astype(np.float64)
    qw = fh.upload_qweight(g, kind, raw, k, n)
    for m in (2, 3, 31, 32, 33, 64):
        x = rng.standard_normal((m, k)).astype(np.float32)
        gx, gy = g.upload(np.concatenate([[0.0], x.reshape(-1)])), g.zeros(m * n)
        fh.linear_q_ptr(g, gx.device_ptr() + 4, qw, gy.device_ptr(), m)
        first = g.read(gy)
        fh.linear_q_ptr(g, gx.device_ptr() + 4, qw, gy.device_ptr(), m)
        got = g.read(gy)
        assert np.array_equal(first.view(np.uint32), got.view(np.uint32)), (kind_name, k, n, m)
        bound = (k + 8) * 2.0**-24 * (np.abs(x).astype(np.float64) @ np.abs(w))
        err = np.abs(got.reshape(m, n) - x.astype(np.float64) @ w)
        assert np.all(err <= bound), (kind_name, k, n, m, float((err / np.maximum(bound, 1e-38)).max()))
    bad = {"Fp8E4M3": [0xff], "Fp8E5M2": [0x7c], "F16": [0x00, 0xfc]}.get(kind_name)
    if bad is None or n < 2:
        return
    nb = raw.size // (k // 32 * n)
    codes = raw.copy().reshape(n, k // 32, nb)
    codes[0, -1, nb - len(bad):] = bad
    codes[-1, 0, nb - 32 if nb == 34 else 0:][: len(bad)] = bad
    qw = fh.upload_qweight(g, kind, codes.reshape(-1), k, n)
    m = 5
    gx, gy = g.upload(rng.standard_normal(m * k).astype(np.float32)), g.zeros(m * n)
    fh.linear_q_ptr(g, gx.device_ptr(), qw, gy.device_ptr(), m)
    nan = np.isnan(g.read(gy).reshape(m, n))
    assert nan[:, [0, -1]].all() and nan.sum() == 2 * m


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0"])
def test_wide_heads_take_the_few_row_kernel(fh, g, orc, kind_name):
    """Products of 17 to 64 rows past 65536 outputs: the few-row kernel's bits for a short K, the ring kernel's for a
    longer one and for one output tile less."""
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(6)
    for k, n, rows, path in ((64, 65537, 17, "Rows"), (64, 65537, 64, "Rows"), (1536, 65540, 32, "Rows"), (64, 65536, 17, "Tiled"),
                             (1568, 65540, 32, "Tiled"), (928, 65540, 33, "Tiled")):
        base = rng.standard_normal((500, k)).astype(np.float32) * np.float32(0.02)
        raw = orc.encode(int(kind), base.reshape(-1)).reshape(500, -1)[np.arange(n) % 500]
        qw, gx = fh.upload_qweight(g, kind, raw.reshape(-1), k, n), g.upload(rng.standard_normal(rows * k).astype(np.float32))
        ya, yb, yc = g.zeros(rows * n), g.zeros(rows * n), g.zeros(rows * n)
        fh.linear_q(g, gx, qw, ya, rows)
        fh.linear_q_with(g, gx, qw, yb, rows, fh.QPath[path])
        fh.linear_q_with(g, gx, qw, yc, rows, fh.QPath["Tiled" if path == "Rows" else "Rows"])
        a, b, c = (g.read(y).view(np.uint32) for y in (ya, yb, yc))
        assert np.array_equal(a, b), (k, n, rows)
        assert not np.array_equal(a, c), (k, n, rows)  # (the other kernel sums in another order)
