"""A decode launch that takes the projections' rows as they are against the launch in front that prepares them (which calls
with biases keep, zeros here): the same bits in the rotated queries, the cache and the result."""
import numpy as np
import pytest

import shainet_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,hd", [(32, 8, 64), (8, 8, 64), (32, 4, 128), (32, 2, 64), (16, 1, 128), (6, 2, 128)])
@pytest.mark.parametrize("norms", ["none", "both", "q", "k"])
@pytest.mark.parametrize("lengths", [[0], [15], [16], [63], [64], [1024], [0, 1, 15, 16, 17, 100]])
def test_rows_prepared_by_the_decode_launch(H, KV, hd, norms, lengths):
    import torch

    assert sa.HIP.fully_available(), "no gfx950 device or libshainet_hip_kernels.so missing"
    gen = torch.Generator(device="cuda").manual_seed(H + hd + len(lengths))
    qn, kn = ((1 + 0.1 * np.random.default_rng(i).standard_normal(hd)).astype(np.float32) if norms in ("both", n) else None
              for i, n in enumerate("qk"))
    B, room = len(lengths), max(lengths) + 5
    q, k, v = (torch.randn((B, n * hd), generator=gen, device="cuda") for n in (H, KV, KV))
    cached = [torch.randn((2, KV, n, hd), generator=gen, device="cuda") if n else None for n in lengths]
    nothing = torch.full((KV, room, hd), float("nan"), device="cuda")
    got = []
    for way in ("fused", "apart", "in place"):
        ctx = sa.AttnContext(H, KV, hd, q_norm=qn, k_norm=kn, eps=1e-6, max_positions=room)
        if way == "apart":
            ctx.set_bias(*(np.zeros(n * hd, np.float32) for n in (H, KV, KV)))
        cache = sa.KVCache(ctx, B, room)
        torch.cuda.synchronize()
        for s, n in enumerate(lengths):  # rows nobody has written yet hold anything
            cache.fill(s, nothing, nothing)
            cache.truncate(s, 0)
            if n:
                cache.fill(s, cached[s][0].contiguous(), cached[s][1].contiguous())
        rows = [q.clone(), k.clone(), v.clone()]
        torch.cuda.synchronize()
        out = rows[0] if way == "in place" else torch.empty_like(q)  # in place: the launch in front again
        for _ in range(3):
            for s, n in enumerate(lengths):
                cache.truncate(s, n)
            if way == "in place":
                ctx.sync()
                rows[0].copy_(q)
                torch.cuda.synchronize()
            ctx.forward(cache, *rows, [1] * B, out=out)
        ctx.sync()
        got.append([out.cpu().numpy(), ctx.last_q_rot(B)]
                   + [x for s, n in enumerate(lengths) for c in range(KV) for x in cache.read(s, c, 0, n + 1)])
    assert np.isfinite(got[0][0]).all()
    for other in got[1:]:
        assert [i for i, (a, b) in enumerate(zip(got[0], other)) if not np.array_equal(a, b)] == []
