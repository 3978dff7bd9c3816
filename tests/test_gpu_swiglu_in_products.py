"""SwiGLU where a product's sums are, without pieces, against 64 bits: every tile that does it, columns that do not fill one, K that
does not fill a step, tiles that two workgroups share, and a tile computed again because a value in it is not finite."""
import numpy as np
import pytest

from test_gpu_bf16_weights import write
from test_gpu_norms_behind_sums import hip, llama, logits_in_64_bits  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("short,T,d,ff,tile,waits", [
    (True, 9, 256, 36, (32, 64), False), (True, 9, 260, 4100, (32, 64), False), (True, 9, 36, 36, (32, 128), False),
    (True, 3000, 64, 132, (64, 128), False), (True, 77, 72, 8196, (96, 128), False), (True, 2000, 36, 516, (128, 256), False),
    (True, 200, 512, 6148, (128, 256), True), (True, 1500, 516, 8196, (256, 256), True), (False, 260, 64, 36, (128, 256), False),
    (False, 200, 516, 8196, (128, 128), True), (False, 1500, 512, 8196, (256, 256), True)])
def test_swiglu_in_the_product(hip, tmp_path, short, T, d, ff, tile, waits):  # noqa: F811
    """Sums of up to 8196 terms round a row by 8196^0.5 times 2^-24 at random, and what they hand on as much again; gate and up of
    different columns make a row of its own."""
    plan = hip.hip.describe_matmul(T, d, 2 * ff, bf16_weights=short)
    assert plan["pieces"] == 1 and plan["tile"] == tile and plan["waits"] == waits, plan
    cfg, w = llama(d, ff, 260, d + T)
    if not short:
        for n in w:
            if w[n].ndim == 2:
                w[n] = w[n] * np.float32(1 + 2.0 ** -12)
    tokens = np.random.default_rng(1).integers(0, 259, T)
    model = hip.HFLoader.load_model(write(tmp_path / "m", cfg, w, lambda n: short, nudge=False))
    got, want = model.run_rows(tokens, range(T)).astype(np.float64), logits_in_64_bits(w, tokens)
    off = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert off.max() <= 2 * 8196 ** 0.5 * 2.0 ** -24, off.max()
    # the last row, which no other one sees, is not a number
    w["model.embed_tokens.weight"][259, d // 2] = np.nan
    tokens[-1] = 259
    model = hip.HFLoader.load_model(write(tmp_path / "n", cfg, w, lambda n: short, nudge=False))
    got = model.run_rows(tokens, range(T)).astype(np.float64)
    assert np.isnan(got[-1]).all()
    off = np.linalg.norm(got - want, axis=1)[:-1] / np.linalg.norm(want, axis=1)[:-1]
    assert off.max() <= 2 * 8196 ** 0.5 * 2.0 ** -24, off.max()
