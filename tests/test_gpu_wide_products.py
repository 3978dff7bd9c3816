"""Products of bf16 weights in tiles of 128 x 256 and 256 x 256, whose steps are 32 of K: one step and two, an odd number of them and an even one,
a last step that is half full (16 of K) and nearly empty (4), rows and columns that end within a block of 16 or within the four or eight
columns of a lane; whole tiles, tiles cut into pieces and tiles that two workgroups share."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,N,tile,pieces,waits", [
    (257, 32, 8204, 128, False, False), (400, 64, 8204, 128, False, False), (777, 1040, 16384, 256, False, False), (513, 100, 32772, 128, False, True),
    (777, 1056, 16388, 128, False, True), (1100, 4096, 1028, 128, True, False), (1100, 4112, 1028, 128, True, False), (1100, 4100, 1028, 128, True, False),
    (2000, 992, 8188, 256, False, False), (2031, 1008, 8188, 256, False, False), (3000, 544, 8204, 256, False, True), (2993, 548, 8204, 256, False, True),
    (2000, 2048, 2308, 256, True, False), (2049, 2100, 2308, 256, True, False)])
def test_wide_products_against_64_bits(T, K, N, tile, pieces, waits):
    """An accumulator rounds three times for 32 terms, and where pieces and the residual are added: (3 K / 32 + 4)^0.5 roundings of 2^-24 at
    random, of sums that are no larger than the last one on average; twice that for the worst row and column."""
    import torch

    import shainet_amd as sa
    from shainet_amd import hip

    assert sa.HIP.fully_available()
    plan = hip.describe_matmul(T, K, N, bf16_weights=True)
    assert (plan["kind"], plan["tile"], plan["pieces"] > 1, plan["waits"]) == ("tiles", (tile, 256), pieces, waits), plan
    assert plan["ragged_k"] == (K % 32 != 0), plan
    g = torch.Generator(device="cuda").manual_seed(T + K + N)
    x = torch.randn((T, K + 4), generator=g, device="cuda")[:, :K]  # (rows of x need not be dense)
    w = torch.randn((K, N), generator=g, device="cuda").bfloat16().float()
    res = torch.randn((T, N), generator=g, device="cuda")
    want = x.double() @ w.double() + res.double()
    for _ in range(2):  # (the second finds the pieces' flags as the first left them)
        got = hip.matmul(x, w, res, bf16_weights=True)
        for dim in (0, 1):
            off = float(((got.double() - want).norm(dim=dim) / want.norm(dim=dim)).max())
            assert off <= 2 * (3 * K / 32 + 4) ** 0.5 * 2.0 ** -24, off


@pytest.mark.parametrize("T,K,N", [(257, 20, 8204), (1300, 28, 16380), (1300, 36, 16380), (257, 48, 8204), (2000, 60, 8188)])
def test_products_that_end_within_their_first_or_second_step(T, K, N):
    test_wide_products_against_64_bits(T, K, N, 128, False, False)


@pytest.mark.parametrize("T,K,N", [(257, 28, 8204), (257, 52, 8204), (777, 1040, 16384), (1100, 4100, 1028), (3000, 548, 8204)])
def test_last_step_and_what_is_not_finite(T, K, N):
    """Values that are not finite, or too large to be lifted, among the last 32 of K, those counted in the last step and those that the step before it
    had: a sum they take part in is what fp32 makes of it, every other one as if they were not there."""
    import torch

    import shainet_amd as sa
    from shainet_amd import hip

    assert sa.HIP.fully_available()
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn((T, K), generator=g, device="cuda")
    w = torch.randn((K, N), generator=g, device="cuda").bfloat16().float()
    for i, value in enumerate([float("inf"), float("nan"), -float("inf"), 2.0 ** 120]):
        k = K - 1 - (9 * i) % min(K, 32)
        x[5 + 50 * i, k] = value
        w[k, 7 + 100 * i] = value
    got = hip.matmul(x, w, bf16_weights=True)
    want = x.cpu().double() @ w.cpu().double()
    got = got.cpu().double()
    finite = want.abs() < 3e38
    assert torch.equal(got[finite].isfinite(), torch.ones(int(finite.sum()), dtype=torch.bool))
    assert torch.equal(got.isnan()[~finite], want.isnan()[~finite]) and not got[~finite].isfinite().any()
    # (K terms of size 1, taken again one after the other, round K^0.5 times at random by 2^-25 of a sum of K^0.5; the worst of 10^7 is 6 of these)
    assert float((got - want)[finite & (want.abs() < 2.0 ** 100)].abs().max()) <= 6 * K * 2.0 ** -24
