"""The ring kernel of the precise GEMM (QPath.Tiled below the streaming kernel's sizes) against the
float64 product of the stored weights, every output held to the summation error bound of any order (as
test_gpu_rows.py: (k + 8) 2^-24 sum_k |x_k w_k|).

Sizes: one block of K and block counts that are not a multiple of the wavefront groups (some groups then
add zeros), fewer than the ring's depth, and deep enough for two K splits that add into y (run twice:
the same bits whichever lands first); 32-row tiles and their edges; columns below, at and past a
wavefront's 64 and the tile's 128; shapes whose plan takes the 64 x 256 tiles. RAGGED: each tile (rows x columns), with
part-filled row and column tiles and odd block counts, by ring_plan on 256 CUs (planes, GGUF rows where another)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RAGGED = [
    (896, 4865, (300,)),    # 64 x 128 (F16 32 x 256)
    (5664, 2047, (290,)),   # 64 x 128, two K splits into y (F16 32 x 128)
    (2080, 11261, (300,)),  # 64 x 256 in three phases, GGUF rows in one
    (1376, 3053, (975,)),   # 64 x 256 in two phases
    (2080, 2563, (513,)),   # 64 x 128, FP8 in two phases (MXFP4 and F16 32 x 256)
    (4896, 897, (1025,)),   # 64 x 128 in two phases (GGUF rows: gemm_ext_kernel)
    (992, 33001, (20,)),    # 32 x 256
]


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
@pytest.mark.parametrize("k,n,rows", [(32, 1, (2, 33)), (96, 65, (31, 32, 33, 65)), (160, 129, (64, 130)),
                                      (512, 300, (5, 40, 129)), (1056, 257, (33, 64, 200)), (4896, 127, (17, 100)),
                                      (896, 9728, (300,)), (2048, 2560, (1024,))] + RAGGED)
def test_ring_product(fh, g, orc, kind_name, k, n, rows):
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(k + n)
    b = orc.quantise_matrix(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32), k, n)
    w = orc.dequantised_in_out(int(kind), b, k, n).reshape(k, n).astype(np.float64)
    qw = fh.upload_qweight(g, kind, b, k, n)
    for m in rows:
        x = rng.standard_normal((m, k)).astype(np.float32)
        gx, gy = g.upload(x), g.upload(np.full(m * n, np.nan, np.float32))
        fh.linear_q_with(g, gx, qw, gy, m, fh.QPath.Tiled)
        first = g.read(gy)
        fh.linear_q_with(g, gx, qw, gy, m, fh.QPath.Tiled)
        got = g.read(gy)
        assert np.array_equal(first.view(np.uint32), got.view(np.uint32)), (kind_name, k, n, m)
        bound = (k + 8) * 2.0**-24 * (np.abs(x).astype(np.float64) @ np.abs(w))
        err = np.abs(got.reshape(m, n) - x.astype(np.float64) @ w)
        worst = float((err / np.maximum(bound, 1e-38)).max())
        print(f"{kind_name} {m} x {k} x {n}: {worst:.3f} of the bound", flush=True)
        assert np.all(err <= bound), (kind_name, k, n, m, worst)


@pytest.mark.parametrize("kind_name", ["Fp8E4M3", "Fp8E5M2", "Fp4", "F16"])
@pytest.mark.parametrize("k,n,rows", [(32, 1, (2, 33)), (96, 65, (31, 33, 65)), (160, 129, (64, 130)),
                                      (1056, 257, (33, 200)), (4896, 127, (17, 100)), (896, 9728, (300,)),
                                      (2048, 2560, (1024,))] + RAGGED)
def test_ring_product_of_gguf_rows(fh, g, orc, kind_name, k, n, rows):
    """The formats kept as GGUF rows: odd block counts put a column's blocks at every byte offset."""
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(k + n)
    raw = orc.encode(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32))
    w = orc.decode(int(kind), raw, k * n).reshape(n, k).T.astype(np.float64)
    qw = fh.upload_qweight(g, kind, raw, k, n)
    for m in rows:
        x = rng.standard_normal((m, k)).astype(np.float32)
        gx, gy = g.upload(x), g.upload(np.full(m * n, np.nan, np.float32))
        fh.linear_q_with(g, gx, qw, gy, m, fh.QPath.Tiled)
        first = g.read(gy)
        fh.linear_q_with(g, gx, qw, gy, m, fh.QPath.Tiled)
        got = g.read(gy)
        assert np.array_equal(first.view(np.uint32), got.view(np.uint32)), (kind_name, k, n, m)
        bound = (k + 8) * 2.0**-24 * (np.abs(x).astype(np.float64) @ np.abs(w))
        err = np.abs(got.reshape(m, n) - x.astype(np.float64) @ w)
        worst = float((err / np.maximum(bound, 1e-38)).max())
        print(f"{kind_name} {m} x {k} x {n}: {worst:.3f} of the bound", flush=True)
        assert np.all(err <= bound), (kind_name, k, n, m, worst)


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("k,n,rows", [(32, 1, (2, 33)), (96, 65, (31, 33, 65)), (160, 129, (64, 130)),
                                      (1056, 257, (33, 200)), (4896, 127, (17, 100)), (896, 9728, (300,)),
                                      (2048, 2560, (1024,))] + RAGGED)
def test_ring_product_of_the_other_paths(fh, g, orc, kind_name, k, n, rows):
    """TiledF16 (x in one f16 part, 11 bits of each element on its row's power-of-two scale: 2^-11 sum_k |x_k w_k|
    beside the summation error; rows up to 1e8) and TiledFast, which takes the precise product here."""
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(k + n)
    b = orc.quantise_matrix(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32), k, n)
    w = orc.dequantised_in_out(int(kind), b, k, n).reshape(k, n).astype(np.float64)
    qw = fh.upload_qweight(g, kind, b, k, n)
    for m in rows:
        x = rng.standard_normal((m, k)).astype(np.float32)
        for path, x, eps in ((fh.QPath.TiledFast, x, 0.0),
                             (fh.QPath.TiledF16, x * (10.0 ** rng.integers(-6, 9, (m, 1))).astype(np.float32), 2.0**-11)):
            gx, gy = g.upload(x), g.upload(np.full(m * n, np.nan, np.float32))
            fh.linear_q_with(g, gx, qw, gy, m, path)
            first = g.read(gy)
            fh.linear_q_with(g, gx, qw, gy, m, path)
            got = g.read(gy)
            assert np.array_equal(first.view(np.uint32), got.view(np.uint32)), (kind_name, path, k, n, m)
            bound = (eps + (k + 8) * 2.0**-24) * (np.abs(x).astype(np.float64) @ np.abs(w))
            err = np.abs(got.reshape(m, n) - x.astype(np.float64) @ w)
            worst = float((err / np.maximum(bound, 1e-38)).max())
            print(f"{kind_name} {path.name} {m} x {k} x {n}: {worst:.3f} of the bound", flush=True)
            assert np.all(err <= bound), (kind_name, path, k, n, m, worst)
