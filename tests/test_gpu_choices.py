"""The largest logit and the largest k where rows end, tie, or hold what is not finite, and where pools of candidates and what a thread
holds of them end."""
import numpy as np
import pytest

from test_gpu_model import INF, NAN, hip, orc  # noqa: F401

pytestmark = pytest.mark.gpu


def rows(vocab):
    r = np.random.default_rng(vocab)
    base = r.standard_normal(vocab).astype(np.float32)
    zeros = np.where(r.random(vocab) < 0.5, np.float32(-0.0), np.float32(0.0))
    ends = np.full(vocab, -1e30, np.float32)
    ends[-1] = -1e29
    odd = base.copy()
    odd[r.integers(0, vocab, vocab // 3 + 1)] = NAN
    odd[r.integers(0, vocab, vocab // 9 + 1)] = INF
    odd[r.integers(0, vocab, vocab // 9 + 1)] = -INF
    crowd = np.round(base)  # (a few values, many times each: pools of any size)
    crowd[r.integers(0, vocab, vocab // 300 + 1)] = 9
    return {"plain": base, "zeros": zeros, "ends": ends, "odd": odd, "crowd": crowd, "nan": np.full(vocab, NAN, np.float32)}


@pytest.mark.parametrize("vocab", [1, 3, 31, 4096, 4099, 32768, 32771, 53250, 65536])
def test_largest_logits(hip, vocab):  # noqa: F811
    d = 8
    m = hip.LlamaModel(vocab, d, 1, 1, 8)
    r = np.random.default_rng(0)
    g = lambda *s: (0.1 * r.standard_normal(s)).astype(np.float32)  # noqa: E731
    m.set_embedding(g(vocab, d))
    m.blocks[0].set_weights(g(d, d), g(d, d), g(d, d), g(d, d))
    m.blocks[0].set_ffn(g(d, 8), g(d, 8), g(8, d))
    m.set_lm_head(g(d, vocab))
    for name, row in rows(vocab).items():
        m.clear_cache()
        m.run([0])
        m.set_logits(row)
        assert m.generate_greedy(1) == [orc.greedy(row)], name
        m.set_logits(row)
        for k in (1, 2, 40, 47, 48, 49, 130):
            ids, vals = hip.Sampler(top_k=k).top_candidates(m)
            want_ids, want_vals = orc.topk(row, k, 1.0)
            np.testing.assert_array_equal(ids, want_ids, f"{name} k={k}")
            np.testing.assert_array_equal(vals.astype(np.float64), want_vals, f"{name} k={k}")
    m.close()
