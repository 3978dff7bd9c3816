"""Rows behind a norm that a product takes as the parts they are the sum of, written so by the norm's own launch or by the one that adds the
pieces of the product in front: numbers whose parts a bf16 holds only when they are lifted, and numbers too large to be lifted, which
stand beside their parts as they are.  A power of two in a norm's weights and its inverse in the columns of the weights behind it
change nothing."""
import numpy as np
import pytest

from test_gpu_bf16_weights import write
from test_gpu_norms_behind_sums import hip, llama, logits_in_64_bits  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,ff,T,tile", [(1024, 4096, 301, (128, 256)), (512, 8196, 1500, (256, 256)), (256, 4096, 399, (128, 256)),
                                         (2048, 2052, 1500, (256, 256))])
@pytest.mark.parametrize("scales", [{}, {7: -112, 9: -120}, {3: 106}, {d: 115 if d % 2 else -115 for d in range(40, 72)}])
def test_rows_as_parts(hip, tmp_path, d, ff, T, tile, scales):  # noqa: F811
    """Sums of up to 8196 terms round a row by 8196^0.5 times 2^-24 at random, those taken again in fp32 every four terms, and what they hand
    on as much again."""
    plan = hip.hip.describe_matmul(T, d, 2 * ff, bf16_weights=True)
    assert plan["kind"] == "tiles" and plan["tile"] == tile, plan
    assert (hip.hip.describe_matmul(T, 1024, d, bf16_weights=True)["pieces"] > 1) == (d in (256, 2048))  # which launch writes them
    cfg, w = llama(d, ff, 260, d + T)
    tokens = np.random.default_rng(1).integers(0, 260, T)
    want = logits_in_64_bits(w, tokens)
    for p in ("model.layers.0.", "model.layers.1."):
        for norm, products in (("input_layernorm", ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj")),
                               ("post_attention_layernorm", ("mlp.gate_proj", "mlp.up_proj"))):
            for column, power in scales.items():
                w[p + norm + ".weight"][column] *= np.float32(2.0 ** power)
                for name in products:
                    w[p + name + ".weight"][:, column] *= np.float32(2.0 ** -power)
    model = hip.HFLoader.load_model(write(tmp_path / "m", cfg, w, lambda n: True, nudge=False))
    got = model.run_rows(tokens, range(T)).astype(np.float64)
    off = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert off.max() <= 2 * 8196 ** 0.5 * 2.0 ** -24, off.max()


@pytest.mark.parametrize("d,ff,T,tile,whole", [(1024, 4096, 301, (128, 256), "pieces"), (512, 8196, 1500, (256, 256), "shared"), (256, 4096, 399, (128, 256), "whole"),
                                               (2048, 2052, 1500, (256, 256), "pieces"), (512, 4096, 700, (128, 256), "shared"), (512, 8192, 2048, (256, 256), "whole")])
@pytest.mark.parametrize("scales", [{}, {7: -112, 9: -120}, {3: 106}])
def test_rows_as_parts_and_as_floats_give_the_same_bits(hip, tmp_path, d, ff, T, tile, whole, scales, monkeypatch):  # noqa: F811
    """Without memory for the parts both launches that write such rows write floats, and a product that reads floats makes the same parts of them itself.
    (A part that is swapped, stale or missing is off by 2^-16 of a number at most: the sums' own rounding covers that.)"""
    plan = hip.hip.describe_matmul(T, d, 2 * ff, bf16_weights=True)
    assert plan["tile"] == tile and whole == ("pieces" if plan["pieces"] > 1 else "shared" if plan["waits"] else "whole"), plan
    cfg, w = llama(d, ff, 260, d + T)
    tokens = np.random.default_rng(1).integers(0, 260, T)
    for p in ("model.layers.0.", "model.layers.1."):
        for column, power in scales.items():
            w[p + "post_attention_layernorm.weight"][column] *= np.float32(2.0 ** power)
            for name in ("mlp.gate_proj", "mlp.up_proj"):
                w[p + name + ".weight"][:, column] *= np.float32(2.0 ** -power)
    folder = write(tmp_path / "m", cfg, w, lambda n: True, nudge=False)
    parts = hip.HFLoader.load_model(folder).run_rows(tokens, range(T))
    monkeypatch.setenv("SHAINET_HIP_TEST_NO_ROWS_AS_PARTS", "1")
    floats = hip.HFLoader.load_model(folder).run_rows(tokens, range(T))
    assert np.isfinite(parts).all() and np.array_equal(parts, floats)
