"""A model's activation arena serves every call of up to the rows it was sized for, and a call of fewer rows may
split its products' K more ways than the largest one: after a long sequence, shorter ones give the bits that a fresh
model gives."""
import numpy as np
import pytest

from oracle import llama_model as lm

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


@pytest.mark.parametrize("path", ["Tiled", "TiledFast", "TiledF16"])
def test_shorter_sequences_after_a_long_one(fh, g, path):
    from ferrum_hip.gguf import Gguf
    from ferrum_hip.llama import GpuLlama

    c = lm.config(vocab=300, ctx=300, dim=512, heads=8, kv_heads=2, head_dim=64, layers=1, hidden=2432, rope_dim=64,
                  rope_base=10000.0, neox=False, eps=1e-5)
    data = lm.to_gguf(lm.llama_random(c, 5, True, False), lm.Q8_0)
    ids = [int(i) for i in np.random.default_rng(1).integers(0, 300, 290)]
    kept = GpuLlama.from_gguf(g, Gguf.parse(data), fh.QPath[path])
    kept.forward_all(ids)
    for t in (1, 33, 64, 96, 100, 129, 160, 224, 260):
        fresh = GpuLlama.from_gguf(g, Gguf.parse(data), fh.QPath[path])
        want = fresh.forward_all(ids[:t])
        got = kept.forward_all(ids[:t])
        assert np.array_equal(np.asarray(got).view(np.uint32), np.asarray(want).view(np.uint32)), (path, t)
