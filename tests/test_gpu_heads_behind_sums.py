"""Heads rotated and put in their places by the launch that adds a product's pieces: small and large heads, rows behind cached ones, odd
numbers of rows, and every way that a tile's registers lie; biases, which take two launches, beside them."""
import numpy as np
import pytest

import refmath as rm
from test_gpu_bf16_weights import write
from test_gpu_model import ATOL, RTOL, _block_calls_match_oracle, _block_pair, _oracle_forward, hip  # noqa: F401
from test_gpu_norms_behind_sums import llama, logits_in_64_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,hd,d,bias,T", [(4, 2, 8, 512, False, 37), (4, 1, 24, 512, False, 21), (8, 2, 64, 1024, False, 50),
                                               (2, 1, 128, 512, False, 21), (8, 2, 64, 1024, True, 50), (8, 2, 12, 512, False, 37)])
def test_heads_of_blocks(hip, H, KV, hd, d, bias, T):  # noqa: F811
    assert hip.hip.describe_matmul(T, d, (H + 2 * KV) * hd)["pieces"] > 1
    _block_calls_match_oracle(hip, d, H, KV, hd, 64, False, bias, [T, 1, T + 2, 3])


@pytest.mark.parametrize("short,T,d,tile", [(True, 33, 516, (32, 64)), (True, 261, 2048, (96, 128)), (True, 513, 1028, (128, 256)),
                                            (True, 1501, 4096, (256, 256)), (False, 261, 516, (128, 256)), (False, 1501, 4096, (256, 256))])
def test_heads_of_every_tile(hip, tmp_path, short, T, d, tile):  # noqa: F811
    """Sums of up to 4096 terms and attention over 1501 rows, sqrt(4096) 2^-24 apart at random and as much again behind them, in two
    blocks; a head in another's place is off by itself."""
    plan = hip.hip.describe_matmul(T, d, 2048, bf16_weights=short)
    assert plan["pieces"] > 1 and plan["tile"] == tile, plan
    cfg, w = llama(d, 64, 260, d + T)
    if not short:
        for n in w:
            if w[n].ndim == 2:
                w[n] = w[n] * np.float32(1 + 2.0 ** -12)
    ids = np.random.default_rng(1).integers(0, 260, T)
    model = hip.HFLoader.load_model(write(tmp_path / "m", cfg, w, lambda n: short, nudge=False))
    got, want = model.run_rows(ids, range(T)).astype(np.float64), logits_in_64_bits(w, ids)
    off = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert off.max() <= 2 * 4096 ** 0.5 * 2.0 ** -24, off.max()


@pytest.mark.parametrize("rows", [50, 17, 3, 1])
def test_a_cache_with_its_lengths_on_the_device_is_refused(hip, rows):  # noqa: F811
    """The block's cache is its caller's, too: while its lengths are on the device a call of any number of rows, whichever launch puts
    them there, would write by the host's old ones.  Nothing is changed by the call that is refused."""
    d, H, KV, hd = 1024, 8, 2, 64
    assert hip.hip.describe_matmul(50, d, (H + 2 * KV) * hd)["pieces"] > 1
    blk, ob, p, r, eps = _block_pair(hip, d, H, KV, hd, 64, 1e6, seed=rows)
    x = r.standard_normal((20, d)).astype(np.float32)
    rm.assert_close(blk.forward_cached(x), _oracle_forward(ob, p, eps, x), ATOL, RTOL, "before")
    lib, cache = hip.hip.lib(), hip.hip.lib().shainet_llama_block_cache(blk._block)
    assert lib.shainet_kv_cache_lengths_to_device(cache) == 0
    x = r.standard_normal((rows, d)).astype(np.float32)
    with pytest.raises(hip.ArgumentError, match="lengths_from_device"):
        blk.forward_cached(x)
    assert lib.shainet_kv_cache_lengths_from_device(cache) == 0
    assert lib.shainet_kv_cache_len(cache, 0) == blk.cache_len == 20
    rm.assert_close(blk.forward_cached(x), _oracle_forward(ob, p, eps, x), ATOL, RTOL, "behind it")
