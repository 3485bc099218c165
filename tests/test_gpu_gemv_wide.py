"""Grouped batch-1 products too wide for the GEMV's LDS records (more than 112 blocks): in a launch of few tasks a task's batches
are shared by a workgroup's four wavefronts. Against the float64 product of the stored weights within the
summation error bound of any order (test_gpu_rows.py), and a plan against the same product alone, bit for
bit. Sizes: the first width past the limit, a last batch of half and of one block, one row, ragged rows,
and more tasks than workgroups fit the chip (a workgroup then streams several)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0"])
def test_wide_plans(orc, kind_name):
    import ferrum_hip as fh

    g = fh.Gpu.open_for_test()
    if g is None:
        pytest.skip("no gfx950 device")
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(4)
    probs, checks, keep = [], [], []
    for k, n in [(3616, 33), (3712, 1), (4864, 896), (5664, 300), (896, 70), (3616, 40000)]:
        base = min(n, 500)  # (rows repeat past 500: the oracle's packing is the slow part)
        b = orc.quantise_matrix(int(kind), (rng.standard_normal(k * base) * 0.02).astype(np.float32), k, base)
        w = orc.dequantised_in_out(int(kind), b, k, base).reshape(k, base).astype(np.float64)
        rows = np.arange(n) % base
        qw = fh.upload_qweight(g, kind, np.asarray(b).reshape(base, -1)[rows], k, n)
        x = rng.standard_normal(k).astype(np.float32)
        gx, gy, gs = g.upload(x), g.zeros(n), g.zeros(n)
        one = fh.GemvPlan(g, [(qw, gx.device_ptr(), gs.device_ptr())])
        one.run()
        probs.append((qw, gx.device_ptr(), gy.device_ptr()))
        checks.append((k, n, gy, gs, (x.astype(np.float64) @ w)[rows], (np.abs(x).astype(np.float64) @ np.abs(w))[rows]))
        keep += [qw, gx, one]
    plan = fh.GemvPlan(g, probs)
    plan.run()
    for k, n, gy, gs, want, mag in checks:
        got = g.read(gy)
        err = np.abs(got - want)
        bound = (k + 8) * 2.0**-24 * mag
        assert np.all(err <= bound), (k, n, float((err / bound).max()))
        assert np.array_equal(got.view(np.uint32), g.read(gs).view(np.uint32)), (k, n)
    plan.free()
    del probs, checks, keep
    g.close()


@pytest.mark.parametrize("kind_name", ["Q8_0", "Q4_0"])
def test_both_kernels_give_the_same_bits(orc, kind_name):
    """A plan of so many tasks that a wavefront takes whole ones, against each product alone, which a workgroup's
    wavefronts share: even and odd batch counts (15, 16, 19, 23), a last half batch and none, ragged rows."""
    import ferrum_hip as fh

    g = fh.Gpu.open_for_test()
    if g is None:
        pytest.skip("no gfx950 device")
    kind = fh.QKind[kind_name]
    rng = np.random.default_rng(9)
    probs, checks, keep = [], [], []
    for k, n in [(3616, 33), (4096, 1), (4864, 896), (3904, 300), (5696, 70), (3840, 64), (3616, 54000)]:
        base = min(n, 300)
        b = orc.quantise_matrix(int(kind), (rng.standard_normal(k * base) * 0.02).astype(np.float32), k, base)
        w = orc.dequantised_in_out(int(kind), b, k, base).reshape(k, base).astype(np.float64)
        rows = np.arange(n) % base
        qw = fh.upload_qweight(g, kind, np.asarray(b).reshape(base, -1)[rows], k, n)
        x = rng.standard_normal(k).astype(np.float32)
        gx, gy, gs = g.upload(x), g.zeros(n), g.zeros(n)
        one = fh.GemvPlan(g, [(qw, gx.device_ptr(), gs.device_ptr())])
        one.run()
        probs.append((qw, gx.device_ptr(), gy.device_ptr()))
        checks.append((k, n, gy, gs, (x.astype(np.float64) @ w)[rows], (np.abs(x).astype(np.float64) @ np.abs(w))[rows]))
        keep += [qw, gx, one]
    plan = fh.GemvPlan(g, probs)
    plan.run()
    for k, n, gy, gs, want, mag in checks:
        got = g.read(gy)
        assert np.all(np.abs(got - want) <= (k + 8) * 2.0**-24 * mag), (k, n)
        assert np.array_equal(got.view(np.uint32), g.read(gs).view(np.uint32)), (k, n)
    plan.free()
    del probs, checks, keep
    g.close()
