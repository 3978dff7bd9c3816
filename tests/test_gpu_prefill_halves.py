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
