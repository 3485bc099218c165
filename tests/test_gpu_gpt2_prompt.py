"""The GPT-2 prompt pass (generate's tokens before the prompt's last one, many rows per product)
against the forward in float64 on the same stored weights, and against one feed per token on a second
copy of the model (held to the CPU oracle by test_gpu_gpt2.py): the next logits after the prompt read
every cache row the pass wrote. The reference's FORWARD tolerance (1e-5, ferrum_wgpu/src/tolerance.rs)
bounds both. The query and key weights are scaled so that scores stay O(1): with the random model's own
(scores of tens, a softmax that picks one key) two f32 forwards drift 1e-5 apart over 500 positions.

Sizes: the fewest tokens the pass takes (6 before the last) and one below; a 32-row tile and past
it; a chunk (512 rows) and past it, with a remainder below the fewest; a start at a position that is
no multiple of 32, so that a query tile's first rows see no key of its last key tile; every head
width the pass takes, both block formats, and head width 256, which stays token by token."""
import numpy as np
import pytest

from oracle import gpt2_model as gm

pytestmark = pytest.mark.gpu
FORWARD = 1e-5


@pytest.fixture(scope="module")
def g():
    import ferrum_hip as fh

    gpu = fh.Gpu.open_for_test()
    if gpu is None:
        pytest.skip("no gfx950 device")
    yield gpu
    gpu.close()


def logits64(m, ids):
    """The last position's logits in float64."""
    d, n, heads = m["dim"], len(ids), m["heads"]
    hd = d // heads
    f = lambda a, *shape: np.asarray(a, np.float64).reshape(*shape)  # noqa: E731

    def norm(x, g, b):
        c = x - x.mean(1, keepdims=True)
        return c / np.sqrt((c * c).mean(1, keepdims=True) + 1e-5) * f(g, -1) + f(b, -1)

    x = f(m["tok"], -1, d)[ids] + f(m["pos"], -1, d)[:n]
    for b in m["blocks"]:
        h = norm(x, b["ln1_g"], b["ln1_b"])
        q, k, v = ((h @ f(b["w" + c], d, d) + f(b["b" + c], -1)).reshape(n, heads, hd).transpose(1, 0, 2) for c in "qkv")
        s = q @ k.transpose(0, 2, 1) / np.sqrt(hd)
        s[:, ~np.tri(n, dtype=bool)] = -np.inf
        p = np.exp(s - s.max(-1, keepdims=True))
        a = (p / p.sum(-1, keepdims=True) @ v).transpose(1, 0, 2).reshape(n, d)
        x = x + a @ f(b["wo"], d, d) + f(b["bo"], -1)
        u = norm(x, b["ln2_g"], b["ln2_b"]) @ f(b["w1"], d, -1) + f(b["b1"], -1)
        x = x + (0.5 * u * (1 + np.tanh(0.7978846 * (u + 0.044715 * u ** 3)))) @ f(b["w2"], -1, d) + f(b["b2"], -1)
    return (norm(x[-1:], m["lnf_g"], m["lnf_b"]) @ f(m["head"], d, -1))[0]


@pytest.mark.parametrize("kind,dim,heads,hidden,layers,before,prompt", [
    ("q8_0", 256, 4, 1024, 3, 0, 6), ("q8_0", 256, 4, 1024, 3, 0, 7), ("q8_0", 256, 4, 1024, 3, 0, 33),
    ("q8_0", 256, 4, 1024, 3, 5, 34), ("q8_0", 256, 4, 1024, 3, 37, 100), ("q8_0", 256, 4, 1024, 3, 3, 513),
    ("q8_0", 256, 4, 1024, 3, 0, 518), ("q8_0", 256, 4, 1024, 3, 0, 520), ("q4_0", 256, 4, 1024, 3, 7, 65),
    ("q4_0", 96, 3, 160, 2, 1, 40), ("q8_0", 64, 8, 96, 2, 2, 70), ("q4_0", 64, 4, 96, 2, 0, 129),
    ("q8_0", 1152, 9, 4128, 2, 11, 50), ("q8_0", 512, 2, 256, 2, 3, 20), ("q8_0", 256, 4, 1024, 1, 0, 20)])
def test_prompt_pass_fills_the_caches_that_feeds_fill(g, kind, dim, heads, hidden, layers, before, prompt):
    from ferrum_hip.gguf import Gguf
    from ferrum_hip.gpt2 import GpuGpt2

    cfg = {"vocab": 500, "ctx": 600, "dim": dim, "heads": heads, "layers": layers, "hidden": hidden}
    model = gm.gpt2_random(cfg, 7)
    for blk in model["blocks"]:
        for name in ("wq", "wk"):
            blk[name] = blk[name] * np.float32(np.sqrt(8.0 / dim))
    data = gm.to_gguf(model, gm.Q8_0 if kind == "q8_0" else gm.Q4_0)
    a, b = GpuGpt2.from_gguf(g, Gguf.parse(data)), GpuGpt2.from_gguf(g, Gguf.parse(data))
    ids = [int(t) for t in np.random.default_rng(prompt).integers(0, cfg["vocab"], before + prompt + 1)]
    for t in ids[:before]:
        a.feed(t, logits=False)
        b.feed(t, logits=False)
    got_pick = a.generate(ids[before:before + prompt], 1)
    assert a.pos() == before + prompt
    for t in ids[before:before + prompt]:
        last = b.feed(t)
    gap = np.sort(last)[-2:]
    if gap[1] - gap[0] > 4 * FORWARD * max(float(np.abs(last).max()), 1.0):
        assert got_pick == [int(np.argmax(last))]
    got, fed, want = a.feed(ids[-1]), b.feed(ids[-1]), logits64(gm.from_gguf(data), ids)
    rel = lambda v: float(np.abs(v - want).max() / max(float(np.abs(want).max()), 1.0))  # noqa: E731
    print(f"{kind} d {dim} heads {heads} positions {before}..{before + prompt}: {rel(got):.2e}, fed {rel(fed):.2e}",
          flush=True)
    assert rel(got) < FORWARD and rel(fed) < FORWARD
    a.free()
    b.free()
