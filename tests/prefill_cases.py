"""The prefill launches whose parity the GPU suite checks at full size, each with the kernel
instantiation the library's own planner picks for it: (head_dim, key chunks merged by the
combine kernel?, wavefront groups, row blocks a workgroup takes in turn), and `+ (True,)` for the
instantiations that run a smaller head_dim in padded tiles.

tests/test_gpu_parity.py runs every case against the oracle on all rows with no tuning
variable set and asserts that the planner's choice is the instantiation named here;
tests/test_prefill_plan_coverage.py (no GPU) asserts that the table still matches the planner
and that every shape of the benchmark configurations, and every instantiation the planner can
reach over a sweep of shapes, is named here."""

# name, H, KV, head_dim, QK-norm, cached positions, new rows, (head_dim, split, groups, turns)
CASES = [
    ("llama1b_prefill_t2048", 32, 8, 64, False, 0, 2048, (64, False, 2, 2)),
    ("llama1b_prefill_t3072", 32, 8, 64, False, 0, 3072, (64, False, 2, 3)),
    ("llama1b_prefill_t8192", 32, 8, 64, False, 0, 8192, (64, False, 1, 0)),
    ("llama1b_prefill_t2560", 32, 8, 64, False, 0, 2560, (64, False, 2, 0)),
    ("llama1b_prefill_t1024", 32, 8, 64, False, 0, 1024, (64, True, 2, 0)),
    ("llama1b_prefill_t45", 32, 8, 64, False, 0, 45, (64, False, 3, 0)),
    ("qwen3_8b_prefill_t45", 32, 8, 128, True, 0, 45, (128, False, 3, 0)),
    ("w1024_chunked_prefill_t2560_on_1000", 16, 2, 64, False, 1000, 2560, (64, True, 3, 0)),
    ("heads64_prefill_t2048", 64, 8, 64, False, 0, 2048, (64, False, 3, 0)),
    ("llama1b_chunked_prefill_t512_on_16384", 32, 8, 64, False, 16384, 512, (64, True, 1, 0)),
    ("qwen3_30b_chunked_prefill_t512_on_16384", 32, 4, 128, True, 16384, 512, (128, True, 1, 0)),
    ("qwen3_30b_chunked_prefill_t512_on_4096", 32, 4, 128, True, 4096, 512, (128, True, 2, 0)),
    ("qwen3_8b_prefill_t2048", 32, 8, 128, True, 0, 2048, (128, False, 2, 2)),
    ("qwen3_8b_prefill_t3072", 32, 8, 128, True, 0, 3072, (128, False, 2, 3)),
    ("qwen3_8b_prefill_t2560", 32, 8, 128, True, 0, 2560, (128, False, 2, 0)),
    ("qwen3_8b_prefill_t4096", 32, 8, 128, True, 0, 4096, (128, False, 1, 0)),
    # head dims below the tile layouts (padded tiles): Phi-3-mini's heads at the bench's size, and smaller ones
    ("phi3_hd96_prefill_t2048", 32, 32, 96, False, 0, 2048, (128, False, 2, 2, True)),
    ("hd96_chunked_prefill_t256_on_8192", 16, 4, 96, True, 8192, 256, (128, True, 2, 0, True)),
    ("hd48_prefill_t8192", 16, 8, 48, False, 0, 8192, (64, False, 1, 0, True)),
    ("hd32_prefill_t1024", 32, 8, 32, True, 0, 1024, (64, True, 2, 0, True)),
]

# The prefill shapes of the benchmark configurations: (H, KV, head_dim, cached positions, new rows).
BASELINE_PREFILL_SHAPES = [
    (32, 8, 64, 0, 2048),
    (32, 8, 64, 0, 8192),
    (32, 4, 128, 16384, 512),
]


def instantiation(plan):
    """The kernel instantiation of a plan dict from shainet_amd.describe_plan."""
    inst = (plan["head_dim"], plan["key_chunks"] > 1, plan["groups"], plan["turns"])
    return inst + (True,) if plan.get("padded") else inst


# Products, each with what the planner runs it as: rows, k, n, (kind, tile, cut into pieces, tiles shared by waiting, k no
# whole number of steps).  Ragged rows and columns where an instantiation is reached with them.
MATMULS = [
    (40, 96, 132, ("few", (32, 128), False, False, False)),
    (33, 100, 260, ("few", (32, 128), False, False, True)),
    (96, 8192, 260, ("few", (32, 128), True, False, False)),
    (70, 2052, 6400, ("few", (32, 128), True, False, True)),
    (200, 512, 16384, ("tiles", (128, 128), False, True, False)),
    (200, 516, 16384, ("tiles", (128, 128), False, True, True)),
    (100, 4096, 3076, ("tiles", (128, 128), True, False, False)),
    (100, 2052, 6400, ("tiles", (128, 128), True, False, True)),
    (1000, 1040, 8192, ("tiles", (128, 256), False, False, False)),
    (1000, 1044, 8192, ("tiles", (128, 256), False, False, True)),
    (1100, 640, 8200, ("tiles", (128, 256), False, True, False)),
    (1100, 644, 8200, ("tiles", (128, 256), False, True, True)),
    (1000, 2048, 2308, ("tiles", (128, 256), True, False, False)),
    (300, 2052, 1028, ("tiles", (128, 256), True, False, True)),
    (2000, 1040, 16384, ("tiles", (256, 256), False, False, False)),
    (2000, 1044, 16384, ("tiles", (256, 256), False, False, True)),
    (3000, 1040, 8200, ("tiles", (256, 256), False, True, False)),
    (3000, 1044, 8200, ("tiles", (256, 256), False, True, True)),
    (1000, 8192, 2308, ("tiles", (256, 256), True, False, False)),
    (1000, 4100, 4092, ("tiles", (256, 256), True, False, True)),
]

# The same of weights that are bf16 numbers: "few" are tiles of 32 to 96 rows whose weights go straight to registers.
BF16_MATMULS = [
    (20, 512, 8196, ("few", (32, 64), False, False, False)),
    (5, 1044, 16380, ("few", (32, 64), False, False, True)),
    (400, 512, 132, ("few", (32, 64), True, False, False)),
    (17, 2052, 132, ("few", (32, 64), True, False, True)),
    (75, 96, 132, ("few", (32, 128), False, False, False)),
    (40, 100, 132, ("few", (32, 128), False, False, True)),
    (5, 512, 132, ("few", (32, 128), True, False, False)),
    (17, 1044, 132, ("few", (32, 128), True, False, True)),
    (97, 96, 8200, ("few", (64, 128), False, False, False)),
    (100, 100, 8196, ("few", (64, 128), False, False, True)),
    (40, 2048, 2308, ("few", (64, 128), True, False, False)),
    (100, 2052, 2308, ("few", (64, 128), True, False, True)),
    (200, 96, 8200, ("few", (96, 128), False, False, False)),
    (200, 100, 8196, ("few", (96, 128), False, False, True)),
    (96, 2048, 3072, ("few", (96, 128), True, False, False)),
    (75, 2052, 2308, ("few", (96, 128), True, False, True)),
    (512, 2048, 16384, ("tiles", (128, 256), False, False, False)),
    (1300, 36, 16380, ("tiles", (128, 256), False, False, True)),
    (400, 640, 8200, ("tiles", (128, 256), False, True, False)),
    (200, 1044, 16384, ("tiles", (128, 256), False, True, True)),
    (1100, 4096, 1028, ("tiles", (128, 256), True, False, False)),
    (1000, 1040, 1028, ("tiles", (128, 256), True, False, True)),
    (300, 1044, 4092, ("tiles", (128, 256), True, False, True)),
    (2000, 640, 8188, ("tiles", (256, 256), False, False, False)),
    (777, 1044, 16384, ("tiles", (256, 256), False, False, True)),
    (3000, 512, 8200, ("tiles", (256, 256), False, True, False)),
    (2000, 2052, 4092, ("tiles", (256, 256), False, True, True)),
    (2000, 2048, 2308, ("tiles", (256, 256), True, False, False)),
    (2000, 4100, 1028, ("tiles", (256, 256), True, False, True)),
]


def matmul_instantiation(plan):
    """The kernel instantiation of a dict from shainet_amd.hip.describe_matmul."""
    return plan["kind"], plan["tile"], plan["pieces"] > 1, plan["waits"], plan["ragged_k"]
