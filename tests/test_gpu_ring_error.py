"""The ring kernel's rounding (QPath.Tiled and AUTO): its plans sum K in chains no longer, in effect, than the K splits of
the tiled kernels make them. The variance of an output's relative error is 0.064 v + 0.58 in units of (1e-7)^2 (F16 0.80), v being the
roundings of f32 sums in units of the last one: nb / (2 parts) for chains of nb / parts blocks, (parts + 1) / 2 -
1 / parts for adding the parts in turn (fitted to products of those kernels, 2% to either side). So the error in the
2-norm against the float64 product stays within 4% of that at the tiled kernels' number of parts. With the fastest plan
instead, the sizes here are 8 to 37% above it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def parts(rows, k, n, planes):
    """K splits of the tiled kernels (gemm_splits over gemm_sum_parts' tiles)."""
    bm = 64 if rows <= (64 if planes else 1024) else 128
    tiles, stages = -(-rows // bm) * -(-n // 128), k // 32
    if tiles >= 512:
        return 1
    return min((-(-tiles * s // 512) * (-(-stages // s) + 2), s) for s in range(1, min(8, max(stages // 4, 1)) + 1))[1]


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0", "Fp8E4M3", "Fp4", "F16"])
@pytest.mark.parametrize("rows,k,n", [(3600, 3808, 736), (2700, 3520, 736), (975, 1344, 3052), (300, 2048, 11264)])
def test_error_of_the_sums(orc, kind_name, rows, k, n):
    import ferrum_hip as fh

    g = fh.Gpu.open_for_test()
    if g is None:
        pytest.skip("no gfx950 device")
    kind, planes = fh.QKind[kind_name], kind_name in ("Q8_0", "Q4_0")
    rng = np.random.default_rng(k)
    raw = orc.encode(int(kind), (rng.standard_normal(k * n) * 0.02).astype(np.float32))
    w = orc.decode(int(kind), raw, k * n).reshape(n, k).T.astype(np.float64)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    qw, gx, gy = fh.upload_qweight(g, kind, raw, k, n), g.upload(x), g.zeros(rows * n)
    fh.linear_q(g, gx, qw, gy, rows)
    got, want = g.read(gy).reshape(rows, n)[:512], x[:512].astype(np.float64) @ w
    p, nb = parts(rows, k, n, planes), k // 32
    v = nb / (2 * p) + (p + 1) / 2 - 1 / p
    bound = 1.04e-7 * np.sqrt(0.064 * v + (0.80 if kind_name == "F16" else 0.58))
    err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    print(f"{kind_name} {rows} x {k} x {n}: {err:.3e}, bound {bound:.3e}", flush=True)
    assert err <= bound
    del qw, gx, gy
    g.close()
