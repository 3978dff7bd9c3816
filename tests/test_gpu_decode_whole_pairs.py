"""Decode attention over pairs of nine tiles and more that are a workgroup's each, the lengths next to them that are cut, and batches of
unequal lengths, against 64 bits."""
import numpy as np
import pytest

import shainet_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,hd,lengths,whole", [
    (32, 8, 64, [16 * 9], True), (32, 8, 64, [16 * 11], True), (8, 8, 64, [16 * 12], False), (8, 2, 32, [16 * 10 + 1], True),
    (32, 8, 64, [16 * 15, 3], True), (16, 8, 64, [16 * 15 + 1, 16 * 15], False), (32, 8, 64, [16 * 9 + 1] + [150] * 15, True),
    (16, 8, 64, [16 * 24] + [1, 17, 130] * 5, True), (16, 8, 64, [16 * 24 + 1] + [380] * 15, False),
    (32, 8, 128, [16 * 16] + [250] * 15, True), (32, 8, 128, [16 * 16 + 1] + [250] * 15, False), (32, 8, 128, [16 * 11], False),
    # a few long pairs among short ones
    (16, 8, 64, [16 * 24] + [16] * 15, False), (16, 8, 64, [16 * 24] + [16 * 8] * 15, False), (16, 8, 48, [16 * 16 + 1] + [9] * 15, False),
    (16, 8, 96, [16 * 16] + [16] * 15, False), (16, 8, 256, [16 * 10] + [16] * 15, False), (16, 8, 128, [16 * 16] + [16] * 31, True)])
def test_decode_over_whole_pairs(H, KV, hd, lengths, whole):
    """A score is a sum of hd products and a result one of up to 385, each rounded by 2^-24: at random 385^0.5 2^-24, 1.2e-6, and
    a score's share, at sizes of up to ten, again."""
    import torch

    assert sa.HIP.fully_available(), "no gfx950 device or libshainet_hip_kernels.so missing"
    B = len(lengths)
    plan = sa.describe_plan(H, KV, hd, [n - 1 for n in lengths], [1] * B)
    assert (plan["units"] == -(-max(lengths) // 16)) == whole, plan
    gen = torch.Generator(device="cuda").manual_seed(sum(lengths))
    q, k, v = (torch.randn((B, n * hd), generator=gen, device="cuda") for n in (H, KV, KV))
    ctx = sa.AttnContext(H, KV, hd, max_positions=max(lengths))
    cache = sa.KVCache(ctx, B, max(lengths))
    old = [torch.randn((2, KV, n - 1, hd), generator=gen, device="cuda") for n in lengths]
    torch.cuda.synchronize()
    for s, n in enumerate(lengths):
        if n > 1:
            cache.fill(s, old[s][0].contiguous(), old[s][1].contiguous())
    out = torch.empty_like(q)
    ctx.forward(cache, q, k, v, [1] * B, out=out)
    ctx.sync()
    turned, out = torch.from_numpy(np.asarray(ctx.last_q_rot(B))).double().reshape(B, H, hd), out.cpu().double().reshape(B, H, hd)
    for s, n in enumerate(lengths):
        for h in range(H):
            c = h * KV // H
            keys, values = (torch.from_numpy(np.asarray(x)).double().reshape(n, hd) for x in cache.read(s, c, 0, n))
            p = torch.softmax(keys @ turned[s, h] / hd ** 0.5, 0)
            want = p @ values
            assert (out[s, h] - want).abs().max() <= 6e-6 * values.abs().max(), (s, h)
