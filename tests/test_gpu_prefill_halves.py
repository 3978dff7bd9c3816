"""Prefill attention in which two groups of wavefronts are half a step apart: one tile of keys and two, a number of tiles that two groups share
unevenly, row blocks that two groups take together where a sequence has an odd number of them or a single one, sequences of
different numbers of blocks whose key chunks are merged by another launch, rows of which only some wavefronts see the last tiles, heads in
padded tiles; operands that are taken again in fp32.  The same where a workgroup is one group with a row block of its own, and batches of sequences
whose layout the planner chooses."""
import pytest

import test_gpu_parity as parity
from test_gpu_parity import hip  # noqa: F401

pytestmark = pytest.mark.gpu

# (cached, new) of each sequence
SEQUENCES = [[(0, 17)], [(0, 32)], [(0, 33)], [(31, 20)], [(0, 65)], [(60, 130)], [(0, 257)], [(5, 300), (0, 40), (200, 129)]]


@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("H,KV,hd", [(2, 2, 64), (8, 2, 64), (4, 1, 128), (3, 3, 128), (2, 1, 96), (4, 2, 36)])
def test_rows_and_tiles_of_two_groups(hip, H, KV, hd, splits, groups, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", str(groups))
    if splits:
        monkeypatch.setenv("SHAINET_HIP_PREFILL_SPLITS", str(splits))
    for n, seqs in enumerate(SEQUENCES):
        ctx, cache, blocks, r = parity.make_pair(hip, H, KV, hd, 1e6, batch=len(seqs), capacity=400, seed=n)
        for s, (cached, _) in enumerate(seqs):
            if cached:
                k, v = (r.standard_normal((KV, cached, hd)).astype("float32") for _ in range(2))
                cache.fill(s, k, v)
                blocks[s].fill_cache(k, v)
        assert parity.check_step(ctx, cache, blocks, r, [new for _, new in seqs], what=str(seqs)) < 1e-4
        cache.close()
        ctx.close()


@pytest.mark.parametrize("hd,KV,T,cached", [(64, 2, 300, 0), (128, 2, 70, 100), (96, 4, 140, 33)])
def test_two_row_blocks_and_what_is_not_finite(hip, hd, KV, T, cached, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", "1")
    parity.test_prefill_keeps_what_is_not_finite(hip, hd, KV, T, cached)


@pytest.mark.parametrize("hd,KV,T,tiny", [(64, 2, 300, 4.70197740328915e-38), (128, 2, 300, 2.2958874039497803e-41)])
def test_two_row_blocks_of_zeros_and_a_tiny_value(hip, hd, KV, T, tiny, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", "1")
    parity.test_prefill_of_zeros_and_a_tiny_value(hip, hd, KV, T, tiny)


@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("H,KV,hd", [(2, 2, 64), (8, 2, 64), (4, 1, 128), (3, 3, 128), (2, 1, 96), (4, 2, 36)])
def test_rows_and_tiles_of_one_group(hip, H, KV, hd, splits, monkeypatch):  # noqa: F811
    test_rows_and_tiles_of_two_groups(hip, H, KV, hd, splits, 3, monkeypatch)


@pytest.mark.parametrize("hd,KV,T,cached", [(64, 2, 300, 0), (128, 2, 70, 100), (96, 4, 140, 33)])
def test_one_group_and_what_is_not_finite(hip, hd, KV, T, cached, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", "3")
    parity.test_prefill_keeps_what_is_not_finite(hip, hd, KV, T, cached)


@pytest.mark.parametrize("hd,KV,T,tiny", [(64, 2, 300, 4.70197740328915e-38), (128, 2, 300, 2.2958874039497803e-41)])
def test_one_group_of_zeros_and_a_tiny_value(hip, hd, KV, T, tiny, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", "3")
    parity.test_prefill_of_zeros_and_a_tiny_value(hip, hd, KV, T, tiny)


# (cached, new) of each sequence; more row blocks than compute units
@pytest.mark.parametrize("H,KV,hd,seqs,groups", [(32, 8, 64, [(0, 40)] * 60, 3), (32, 32, 96, [(0, 100), (30, 40)] * 13, 3), (8, 8, 128, [(0, 90 + i) for i in range(50)], 3),
                                                 (32, 8, 64, [(700, 40)] * 50, 1)])
def test_many_sequences_as_planned(hip, H, KV, hd, seqs, groups):  # noqa: F811
    plan = hip.describe_plan(H, KV, hd, [c for c, _ in seqs], [n for _, n in seqs])
    assert plan["groups"] == groups, plan
    ctx, cache, blocks, r = parity.make_pair(hip, H, KV, hd, 1e6, batch=len(seqs), capacity=800, seed=1)
    for s, (cached, _) in enumerate(seqs):
        if cached:
            k, v = (r.standard_normal((KV, cached, hd)).astype("float32") for _ in range(2))
            cache.fill(s, k, v)
            blocks[s].fill_cache(k, v)
    assert parity.check_step(ctx, cache, blocks, r, [new for _, new in seqs], what=str(seqs[:2])) < 1e-4
    cache.close()
    ctx.close()


@pytest.mark.parametrize("groups", [1, 2, 3])
@pytest.mark.parametrize("hd,KV,T,cached", [(64, 2, 300, 0), (96, 4, 40, 33), (128, 2, 70, 100)])
def test_scores_keep_all_24_bits_in_every_layout(hip, hd, KV, T, cached, groups, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", str(groups))
    parity.test_prefill_scores_keep_all_24_bits(hip, hd, KV, T, cached)


@pytest.mark.parametrize("groups", [1, 2, 3])
@pytest.mark.parametrize("of_keys", [False, True])
@pytest.mark.parametrize("hd,KV,T,splits", [(16, 2, 300, 0), (64, 2, 300, 3), (64, 8, 2300, 0), (96, 2, 300, 0), (128, 2, 300, 0), (128, 8, 2300, 0)])
def test_third_parts_in_every_layout(hip, hd, KV, T, splits, of_keys, groups, monkeypatch):  # noqa: F811
    """One operand is 1 + 2^-9 + 0.9 x 2^-17 in its even elements, of which the last summand is a bf16 part of its own, the other 1 and
    -(1 + 2^-9) by turns: what is left of the scores of even keys, 2^18 times 0.9 x 2^-17, comes from third parts alone.  The odd keys have
    the same score from one product of two leading parts.  A result is a difference of the weights of both, the bound what six products
    leave out, the sums and the factor of the queries: 2^-23 of the sum of the products' sizes, 2^19, in log2 units.  2300 rows of 8 heads are
    more workgroups than compute units: nothing pads their LDS."""
    import numpy as np
    import torch

    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", str(groups))
    if splits:
        monkeypatch.setenv("SHAINET_HIP_PREFILL_SPLITS", str(splits))
    H, third = 2 * KV, 0.9 * 2.0 ** -17
    c = float(np.float32(np.log2(np.e)) * np.float32(1 / np.sqrt(hd)))
    size = 2.0 ** (13 - int(np.log2(hd)))
    long, short = np.ones(hd), np.ones(hd)
    long[0::2] = 1 + 2.0 ** -9 + third
    short[1::2] = 1 + 2.0 ** -9
    query, key = (short, long) if of_keys else (long, short)
    key[1::2] *= -1
    odd_key = np.zeros(hd)
    odd_key[1] = hd / 2 * third
    q = torch.tensor(np.tile(2.0 ** 6 / c * query, (T, H)), dtype=torch.float32, device="cuda")
    keys = torch.tensor(np.where(np.arange(T)[:, None] % 2, odd_key, key) * size, dtype=torch.float32, device="cuda")
    values = torch.ones((T, hd), device="cuda")
    values[1::2] = -1
    ctx = hip.AttnContext(H, KV, hd, rope_freqs=np.zeros(hd // 2, np.float32), max_positions=T)
    torch.cuda.synchronize()
    cache = hip.KVCache(ctx, 1, T)
    ctx.sync()
    got = ctx.forward(cache, q, keys.repeat(1, KV), values.repeat(1, KV), [T])
    ctx.sync()
    got = got.cpu().numpy().reshape(T, H, hd).astype(np.float64)
    s = keys.cpu().numpy().astype(np.float64) @ q[0, :hd].cpu().numpy().astype(np.float64) / np.sqrt(hd)  # every row's, every head's
    sizes = float(np.abs(keys[0].cpu().numpy().astype(np.float64)) @ q[0, :hd].cpu().numpy().astype(np.float64) / np.sqrt(hd))
    even, odd = np.exp(s[0] - s[:2].max()) * (np.arange(T) // 2 + 1), np.exp(s[1] - s[:2].max()) * ((np.arange(T) + 1) // 2)
    bound = 0.5 * 2.0 ** -23 * sizes + 1e-5
    assert 0.5 * (1 - np.exp(-abs(s[0]))) > 8 * bound  # (without those parts an even key's score is 0)
    assert np.abs(got - ((even - odd) / (even + odd))[:, None, None]).max() <= bound
    cache.close()
    ctx.close()


@pytest.mark.parametrize("groups", [1, 2, 3])
@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("name", ["even", "narrow_values", "wide_values", "large"])
def test_values_by_distance_in_every_layout(hip, tmp_path, name, splits, groups, monkeypatch):  # noqa: F811
    """290 rows of one and of two heads a key's: 3 and 5 row blocks, rows on both sides of the table's reach."""
    import numpy as np
    import test_gpu_zabutar as zabutar

    monkeypatch.setenv("SHAINET_HIP_PREFILL_GROUPS", str(groups))
    if splits:
        monkeypatch.setenv("SHAINET_HIP_PREFILL_SPLITS", str(splits))
    cfg, rows = zabutar.attention_config(name)
    p = zabutar.Pair(hip, tmp_path, cfg, rel_rows=rows)
    x = np.random.default_rng(5).standard_normal((290, cfg["width"])).astype(np.float32)
    want, b = p.layer(0, x), p.model.blocks[0]
    zabutar.close(b.forward_cached(x), want)
    zabutar.close(zabutar.block_cut(b, x, (33, 257)), want)


@pytest.mark.parametrize("H,KV,hd,T,cached,chain", [(32, 8, 64, 400, 4000, 35), (32, 8, 64, 300, 8000, 44), (32, 8, 64, 800, 4000, 30), (32, 4, 128, 512, 4096, 36),
                                                    (32, 8, 96, 300, 4000, 23)])
def test_long_chains_are_rounded_once_a_tile(hip, H, KV, hd, T, cached, chain):  # noqa: F811
    """chain: tiles that one group of wavefronts walks through, as planned.  A result is the sum of as many, rounded once for each (2^-24 of it at
    most, at random), and comes from scores whose errors move it by four times that at most: the root of the sum of squares."""
    import torch

    plan = hip.describe_plan(H, KV, hd, [cached], [T])
    tiles = -(-(-(-(cached + T) // 32)) // plan["key_chunks"])
    assert plan["groups"] in (2, 3) and -(-tiles // (2 if plan["groups"] == 2 else 1)) == chain, plan
    S, g = cached + T, H // KV
    r = torch.Generator(device="cuda").manual_seed(hd + T)
    q, k, v = (torch.randn((T, n * hd), generator=r, device="cuda") for n in (H, KV, KV))
    kc, vc = (torch.randn((KV, cached, hd), generator=r, device="cuda") for _ in range(2))
    ctx = hip.AttnContext(H, KV, hd, max_positions=S)
    torch.cuda.synchronize()
    cache = hip.KVCache(ctx, 1, S)
    cache.fill(0, kc, vc)
    ctx.sync()
    got = ctx.forward(cache, q, k, v, [T])
    ctx.sync()
    got = got.double().reshape(T, H, hd)
    qr = torch.tensor(ctx.last_q_rot(T), device="cuda").double().reshape(T, H, hd)
    hidden = torch.arange(S, device="cuda")[None] > cached + torch.arange(T, device="cuda")[:, None]
    off = size = 0.0
    for h in range(0, H, g):  # one head of each group
        kr, vr = (torch.tensor(a, device="cuda").double() for a in cache.read(0, h // g, 0, S))
        s = (qr[:, h] @ kr.T.contiguous() / hd ** 0.5).masked_fill(hidden, float("-inf"))
        want = torch.softmax(s, -1) @ vr
        off += ((got[:, h] - want) ** 2).sum().item()
        size += (want ** 2).sum().item()
    assert (off / size) ** 0.5 <= 2.0 ** -24 * (chain + 16) ** 0.5, ((off / size) ** 0.5, 2.0 ** -24 * (chain + 16) ** 0.5)
    cache.close()
    ctx.close()
