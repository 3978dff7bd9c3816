"""No GPU: the planner's choice of prefill kernel for every benchmark shape, and for a sweep of
other shapes, is an instantiation that a full-size GPU parity case names (tests/prefill_cases.py),
so that a change of the planner cannot move a configuration onto an untested kernel unnoticed."""
import itertools

import prefill_cases as pc
import shainet_amd as sa


def plan_of(H, KV, hd, S, T):
    return sa.describe_plan(H, KV, hd, [S], [T])


def test_cases_name_the_planners_choice():
    for name, H, KV, hd, _norm, S, T, inst in pc.CASES:
        plan = plan_of(H, KV, hd, S, T)
        assert plan["path"] == sa.hip.PATH_PREFILL, name
        assert pc.instantiation(plan) == inst, (name, plan)


def test_every_benchmark_prefill_shape_is_a_case_at_full_size():
    shapes = {(H, KV, hd, S, T) for _, H, KV, hd, _, S, T, _ in pc.CASES}
    for shape in pc.BASELINE_PREFILL_SHAPES:
        assert shape in shapes, shape


def test_bench_prefill_workloads_are_cases():
    # bench.py's prefill workloads (name -> shape) against the table: the bench times nothing
    # whose output no test has looked at
    import bench

    by_name = {name: (H, KV, hd, S, T) for name, H, KV, hd, _, S, T, _ in pc.CASES}
    for name, H, KV, hd, _theta, _norm, lens, T in bench.PREFILL_WORKLOADS:
        if lens is not None and len(lens) == 1:
            assert by_name.get(name) == (H, KV, hd, lens[0], T), name


def test_every_reachable_instantiation_is_covered():
    # (the instantiations for padded tiles, a fifth element in the table, are the same code with the
    # head_dim of the data as a run-time value; the table holds four of them, both tile widths, with
    # and without key chunks, turns and one workgroup per block, and this sweep does not enumerate them)
    covered = {inst for *_, inst in pc.CASES if len(inst) == 4}
    seen = set()
    for hd, KV, g in itertools.product((64, 128), (1, 2, 4, 8), (1, 2, 4, 8)):
        for S in (0, 1000, 4096, 16384, 32768):
            for T in (17, 64, 100, 128, 256, 300, 512, 768, 1024, 1536, 2048, 2560, 3072, 4096, 6144, 8192):
                plan = plan_of(KV * g, KV, hd, S, T)
                if plan["path"] != sa.hip.PATH_PREFILL:
                    continue
                seen.add(pc.instantiation(plan))
    assert seen <= covered, sorted(seen - covered)
    assert seen == covered, sorted(covered - seen)  # and nothing in the table is unreachable


def test_batches_of_short_sequences_have_a_group_for_each_row_block():
    # two row blocks a workgroup only where they fill it, and where the keys are many enough for that to be worth a compute unit's wait for its next one
    for H, KV, hd, B, cached, new, groups in [
            (32, 8, 64, 64, 0, 40, 3), (32, 8, 64, 64, 0, 200, 3), (32, 8, 64, 48, 0, 65, 3), (32, 8, 64, 8, 16384, 32, 3),
            (32, 8, 128, 8, 16384, 32, 3), (32, 32, 96, 25, 0, 100, 3), (32, 32, 96, 64, 500, 40, 3), (32, 32, 128, 64, 2000, 100, 3),
            (32, 8, 64, 64, 500, 40, 1), (32, 8, 64, 64, 2000, 100, 1), (32, 8, 128, 64, 500, 100, 1), (32, 8, 64, 1, 0, 4096, 1)]:
        plan = sa.describe_plan(H, KV, hd, [cached] * B, [new] * B)
        assert plan["groups"] == groups, (H, KV, hd, B, cached, new, plan)
        blocks = B * -(-new * (H // KV) // 128)
        pairs = B * -(-new * (H // KV) // 256)
        assert plan["workgroups"] == (blocks if groups == 3 else pairs) * KV * plan["key_chunks"], plan


def test_few_rows_on_many_are_cut_into_more_chunks():
    # the launch that merges them is short: one chunk more costs it half as much as of many rows
    for cached, new, chunks in [(2000, 17, 8), (2000, 40, 8), (8000, 40, 16), (2000, 200, 4), (4000, 400, 2)]:
        assert sa.describe_plan(32, 8, 64, [cached], [new])["key_chunks"] == chunks, (cached, new)


def test_short_ranges_are_not_shared_by_two_groups():
    for H, KV, hd, B, cached, new, groups in [
            (32, 8, 64, 1, 0, 45, 3), (32, 8, 64, 1, 0, 128, 3), (32, 8, 64, 1, 0, 129, 2), (32, 8, 64, 1, 80, 45, 3), (32, 8, 64, 1, 90, 45, 2),
            (32, 8, 128, 1, 0, 96, 3), (32, 8, 128, 1, 0, 97, 2), (32, 8, 64, 16, 0, 100, 3), (32, 8, 64, 8, 0, 256, 3), (32, 8, 64, 8, 0, 300, 2),
            (32, 8, 128, 16, 0, 100, 3), (32, 8, 64, 1, 2000, 40, 2)]:
        plan = sa.describe_plan(H, KV, hd, [cached] * B, [new] * B)
        assert plan["groups"] == groups, (H, KV, hd, B, cached, new, plan)


def test_chunks_of_heads_over_64_stay_with_a_row_block_a_workgroup():
    # two row blocks a workgroup round a chain of sums six times a tile: only where ranges are long enough for 1024 blocks and chunks, as ever
    for hd, (H, KV), S, T in itertools.product((96, 128), ((32, 8), (32, 4), (16, 8), (8, 8), (24, 4)), (0, 200, 1000, 3000, 6000, 12000),
                                               (40, 100, 200, 400, 700, 1000, 1200, 1500, 2000, 2500)):
        plan = plan_of(H, KV, hd, S, T)
        if plan["path"] != sa.hip.PATH_PREFILL or plan["key_chunks"] == 1:
            continue
        blocks = -(-T * (H // KV) // 128) * KV
        long = -(-(S + T) // 32) // -(-1024 // blocks) >= 32
        assert long or blocks * plan["key_chunks"] <= 768 and plan["groups"] != 1, (hd, H, KV, S, T, plan)


def test_decode_and_generic_paths_are_told_apart():
    assert sa.describe_plan(32, 8, 128, [5000] * 16, [1] * 16)["path"] == sa.hip.PATH_DECODE
    assert sa.describe_plan(32, 8, 128, [5000] * 16, [8] * 16)["path"] == sa.hip.PATH_DECODE  # two entries each
    assert sa.describe_plan(32, 8, 128, [5000] * 16, [9] * 16)["path"] == sa.hip.PATH_PREFILL
    # head dimensions between the tile layouts run in padded tiles: 8 in tiles of 64, 96 in tiles of 128
    small = sa.describe_plan(8, 4, 8, [0], [6])
    assert small["path"] == sa.hip.PATH_DECODE and small["head_dim"] == 64
    assert sa.describe_plan(32, 8, 96, [0], [300])["path"] == sa.hip.PATH_PREFILL
    assert sa.describe_plan(32, 8, 96, [0], [300])["head_dim"] == 128
    assert sa.describe_plan(16, 4, 256, [4096], [1])["head_dim"] == 256
    # what no tile layout holds: not a multiple of 4, or more than 16 rows x heads of head_dim above 128
    assert sa.describe_plan(8, 4, 6, [0], [6])["path"] == sa.hip.PATH_GENERIC
    assert sa.describe_plan(16, 4, 256, [0], [40])["path"] == sa.hip.PATH_GENERIC
    head = sa.describe_plan(32, 8, 128, [5000] * 16, [1] * 16)
    assert head["workgroups"] == 256 and head["units"] * 256 >= 16 * 8 * 313


def test_decode_spans_end_with_the_pairs():
    def split(lens, KV=8, hd=64):
        p = sa.describe_plan(4 * KV, KV, hd, [n - 1 for n in lens], [1] * len(lens))
        return p["workgroups"], p["units"]

    apart = 0
    for tiles in range(1, 250):  # one sequence: spans that end with the pairs, or spans end to end
        wgs, q = split([16 * tiles])
        per = -(-tiles // q)
        if wgs != 8 * per:
            apart += 1
            assert wgs == -(-8 * tiles // q) and q == max(4, -(-8 * tiles // 256)), tiles
        else:  # (all pairs' last spans meet on one XCD only where a span is a tile per wavefront)
            assert per == 1 or per % 8 or q == 4, tiles
    assert apart < 25  # of 249, the most of them long ones
    assert split([16 * 5]) == (8, 5) and split([16 * 8]) == (8, 8)      # whole pairs
    assert split([16 * 12]) == (24, 4) and split([16 * 13]) == (32, 4)
    assert split([16 * 40]) == (80, 4) and split([16 * 32]) == (64, 4)
    assert split([16 * 32] * 2) == (112, 5)   # eight spans each would end on one XCD
    assert split([16 * 24] * 2) == (96, 4) and split([16 * 24] * 4) == (192, 4)
    assert split([16 * 40] * 4) == (224, 6) and split([16 * 16] * 4) == (96, 6)
    assert split([16 * 5] * 16) == (128, 5)
    assert split([16 * 9] * 16) == (231, 5)  # two spans each would meet on four XCDs: 1152 tiles end to end
    assert split([64], 300, 256) == (240, 5)  # more pairs than workgroups: end to end


def test_products_run_as_their_cases_say():
    plan = sa.hip.describe_matmul
    for cases, bf16 in ((pc.MATMULS, False), (pc.BF16_MATMULS, True)):
        for T, K, N, inst in cases:
            assert pc.matmul_instantiation(plan(T, K, N, bf16)) == inst, (T, K, N, plan(T, K, N, bf16))
        seen = set()
        for T, K, N in itertools.product((5, 17, 40, 96, 97, 128, 200, 256, 257, 512, 777, 1024, 1300, 2048, 2304, 3000, 4096),
                                         (4, 32, 100, 512, 1024, 2048, 2052, 4100, 8192), (4, 132, 1024, 2308, 3072, 8192, 16384)):
            seen.add(pc.matmul_instantiation(plan(T, K, N, bf16)))
        assert seen <= {inst for *_, inst in cases}, sorted(seen - {inst for *_, inst in cases})
        assert plan(100, 6, 8, bf16)["kind"] == plan(100, 8, 6, bf16)["kind"] == "plain"


def test_large_tiles_fill_their_last_round():
    # more than a round of 256 tiles of 256 x 256: the last round is empty or at least half full
    for rows in range(2049, 8193, 256):
        tiles = -(-rows // 256) * 32
        plan = sa.hip.describe_matmul(rows, 2048, 8192)
        large = tiles >= 256 and (tiles % 256 == 0 or tiles % 256 >= 128)
        assert (plan["tile"] == (256, 256)) == (large and -(-rows // 256) * 256 * 100 <= -(-rows // 128) * 128 * 115), (rows, plan)


def test_low_tiles_of_bf16_weights_stay_within_a_round():
    # more than a workgroup a compute unit, each with a start of its own, takes up to three times as long as the large tiles
    for T, K, N in ((4000, 32, 4096), (512, 64, 32000), (777, 128, 16384), (2048, 128, 4096), (512, 256, 16384), (1100, 192, 4096)):
        assert sa.hip.describe_matmul(T, K, N, bf16_weights=True)["kind"] == "tiles", (T, K, N)
    for T, K, N in itertools.product((257, 300, 512, 777, 1100, 2048, 4000), (32, 100, 256, 512, 1024, 2048), (132, 1024, 4092, 16384)):
        plan = sa.hip.describe_matmul(T, K, N, bf16_weights=True)
        assert plan["kind"] == "tiles" or plan["workgroups"] <= 256, (T, K, N, plan)


def test_a_few_long_pairs_are_cut():
    """A batch of which some sequences are longer: whole pairs would have their workgroups work alone for the longest.  Where no cut
    ends with the pairs the longest are whole."""
    def split(lens, hd, KV=8, g=4):
        p = sa.describe_plan(g * KV, KV, hd, [16 * n - 1 for n in lens], [1] * len(lens))
        return p["workgroups"], p["units"]

    for hd in (16, 48, 64):
        assert split([24] + [1] * 15, hd) == (160, 5) and split([24] + [8] * 15, hd) == (144, 8)
        assert split([16] + [1] * 15, hd) == (128, 16) and split([24] + [12] * 15, hd) == (128, 24)
        assert split([24] * 4 + [8] * 12, hd) == (192, 8) and split([24] + [1] * 15, hd, g=8) == (128, 24)
    for hd in (96, 128, 256):
        assert split([16] + [1] * 15, hd) == (144, 6) and split([10] + [1] * 15, hd) == split([12] + [4] * 15, hd) == (144, 4)
        assert split([16] + [8] * 15, hd) == (128, 16) and split([16] * 16, hd) == (128, 16) and split([16] + [1] * 31, hd) == (256, 16)
    assert split([16] + [1] * 15, 128, g=8) == (128, 16) and split([16] + [1] * 15, 256, g=8) == (144, 6)
    assert split([24] + [1, 2, 9] * 5, 64) == (128, 24)   # nothing that ends with all of them
    assert split([3] * 16, 64) == (128, 4)


def test_products_of_few_long_sums_stay_in_small_tiles():
    """The larger tiles' sums are longer, and their errors twice as large: a tile of the small ones that is within its bounds is taken
    where the best one by the estimate is not, up to a quarter behind it."""
    def tile(*shape):
        p = sa.hip.describe_matmul(*shape, bf16_weights=True)
        return p["kind"], p["tile"], p["pieces"]

    for T, K, N in ((512, 2048, 1024), (480, 2048, 1024), (1024, 2048, 512), (1000, 2048, 512)):
        assert tile(T, K, N) == ("few", (64, 128), 4)
    for T, K, N in ((777, 1536, 1536), (512, 1536, 2304), (257, 1280, 4608), (3000, 1536, 512)):
        assert tile(T, K, N) == ("few", (96, 128), 2)
    for T, K, N in ((1400, 2048, 260), (257, 2048, 1616), (1700, 8192, 64), (3000, 4096, 64)):
        assert tile(T, K, N)[:2] == ("few", (32, 64))
    for T, K, N in ((600, 1280, 1616), (224, 1280, 4608)):
        assert tile(T, K, N) == ("few", (32, 128), 1)
    assert tile(1000, 1280, 2304)[0] == tile(512, 2048, 2052)[0] == "tiles"   # none that fits


def test_no_more_rows_than_a_grid_has_are_cut_into_pieces():
    """The kernel that adds the pieces has a row per workgroup of its grid's second dimension, which ends at 65535."""
    for T, K, N, bf16 in itertools.product((65536, 65537, 100000, 131072, 500000, 1 << 21), (4, 64, 100, 1024, 8192, 32768),
                                           (4, 32, 100, 132, 512, 1024, 3072, 16384), (False, True)):
        assert sa.hip.describe_matmul(T, K, N, bf16_weights=bf16)["pieces"] == 1, (T, K, N, bf16)


def test_ragged_k_is_told_by_the_steps_of_the_kernel():
    # large tiles take 32 of K at a time where the weights are bf16 numbers, 16 where they are not
    for T, N in ((512, 16384), (2000, 8188), (777, 3072), (3000, 8204)):
        for K in (1008, 1024, 1040, 1044, 4112):
            for bf16, step in ((True, 32), (False, 16)):
                plan = sa.hip.describe_matmul(T, K, N, bf16)
                assert plan["kind"] == "tiles" and plan["ragged_k"] == (K % step != 0), (T, K, N, bf16, plan)
