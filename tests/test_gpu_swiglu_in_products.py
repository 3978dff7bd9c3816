"""SwiGLU where a product's sums are, without pieces, against 64 bits: every tile that does it (and those of 256 x 256 and three parts,
which leave it to a launch of its own), columns that do not fill one, K that
does not fill a step, tiles that two workgroups share, and a tile computed again because a value in it is not finite; and the activation by
itself, in its last bit and far out."""
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
    """Sums of up to max(d, ff) terms round a row by that^0.5 times 2^-24 at random, and what they hand on as much again; gate and up of
    different columns make a row of its own."""
    most = 2 * max(d, ff) ** 0.5 * 2.0 ** -24
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
    assert off.max() <= most, off.max()
    # the last row, which no other one sees, is not a number
    w["model.embed_tokens.weight"][259, d // 2] = np.nan
    tokens[-1] = 259
    model = hip.HFLoader.load_model(write(tmp_path / "n", cfg, w, lambda n: short, nudge=False))
    got = model.run_rows(tokens, range(T)).astype(np.float64)
    assert np.isnan(got[-1]).all()
    off = np.linalg.norm(got - want, axis=1)[:-1] / np.linalg.norm(want, axis=1)[:-1]
    assert off.max() <= most, off.max()


def in_double(gate, up):
    with np.errstate(all="ignore"):
        g = gate.astype(np.float64)
        return ((g / (1 + np.exp(-g))) * up.astype(np.float64)).astype(np.float32)


def near_ties(r, count):
    """Pairs whose silu(gate) up lies 2^-50.5 to 2^-46.5 of its value from the middle between two fp32 numbers: 64 bits of silu times the 24
    of an up, of which those behind the result's 24 are near the half of them.  An activation that is good to 2^-46 gets many of
    them wrong; fp64 with a handful of roundings, 2^-51 together, none."""
    gates, ups = [], []
    up = np.arange(15 << 20, 1 << 24, dtype=np.uint64)
    while len(gates) < count:
        g = np.float32(r.uniform(-30, 30))
        bits = np.uint64(np.ldexp(abs(np.frexp(np.longdouble(g) / (1 + np.exp(-np.longdouble(g))))[0]), 64))
        if bits < np.uint64(0x8fffffffffffffff):
            continue                                        # (the product has 87 bits, not 88)
        near = np.flatnonzero(bits * up - np.uint64((1 << 63) - (1 << 42)) < np.uint64(1 << 43))
        for m in up[near]:
            product = int(bits) * int(m)
            off = np.log2(abs((product & ((1 << 64) - 1)) - (1 << 63)) / product)
            if -50.5 < off < -46.5:
                gates.append(g)
                ups.append(np.float32(int(m) * 2.0 ** -23) * np.float32(r.choice([-1, 1])))
    return np.array(gates[:count], np.float32), np.array(ups[:count], np.float32)


@pytest.mark.parametrize("T", [1, 4, 40, 300])
def test_the_activation_itself(hip, T):  # noqa: F811
    """A block whose attention adds nothing, rows with one value that is 16 behind their norm, and a down product that changes nothing:
    what comes out are the activations of the gates and ups in the weights, the nearest fp32 numbers to what they are in 64 bits and,
    far out and where they are not finite, what fp64 has."""
    d = 256
    r = np.random.default_rng(7)
    gates = r.uniform(-70, 120, (d, d)).astype(np.float32)
    size = np.abs(in_double(gates, np.float32(1)))
    ups = (np.exp2(np.clip(-np.floor(np.log2(size)), -20, 100)) * r.uniform(1, 2, (d, d)) * r.choice([-1, 1], (d, d))).astype(np.float32)
    gates[0], ups[0] = near_ties(r, d)
    inf, big = np.float32(np.inf), np.float32(2.0 ** 100)
    far = [(99.5, 1.5), (-99.5, big), (700.1, 1.1), (-700.1, big), (709.78271, -3), (-709.78271, big), (-709.7828, big), (-760, 3), (760, 3), (1e30, 1e-9),
           (-1e30, 1e30), (3e38, 1e-3), (-3e38, 3), (-0.0, 3), (0.0, -3)]
    gates[1, 2:2 + len(far)], ups[1, 2:2 + len(far)] = np.float32(far).T
    alone = [(inf, 2), (-inf, 2), (inf, 0), (-705, inf), (-709.7828, inf), (3, -inf), (0, inf), (inf, -inf)]   # (a row of its own each)
    for i, pair in enumerate(alone):
        gates[2 + i, 2 + i], ups[2 + i, 2 + i] = pair
    w = [np.clip(a, -3e38, 3e38).astype(np.float32) for a in (gates, ups)]
    w = [np.where(np.isinf(a), b, a / np.float32(16)) for a, b in zip((gates, ups), w)]   # (16 times 3e38 is not finite)
    blk = hip.LlamaBlock(d, 4, d, eps=0.0)
    blk.set_weights(*(np.zeros((d, d), np.float32) for _ in range(4)))
    blk.set_norms(np.ones(d, np.float32), np.ones(d, np.float32))
    blk.set_ffn(*w, np.eye(d, dtype=np.float32))
    finite = np.isfinite(gates) & np.isfinite(ups)
    finite[1] = False
    with np.errstate(all="ignore"):
        exact = np.longdouble(gates) / (1 + np.exp(-np.longdouble(gates))) * np.longdouble(ups)
        want = np.where(finite, exact.astype(np.float32), in_double(gates, ups))
    for first in range(0, 10, T):
        at = np.arange(first, first + T) % d
        x = np.zeros((T, d), np.float32)
        x[np.arange(T), at] = 16
        got = blk.forward(x) - x
        for t, k in enumerate(at):
            own = 2 <= k < 2 + len(alone)
            columns = [k] if own else [c for c in range(d) if c != k]   # (16 and a value are one number)
            assert np.array_equal(got[t, columns], want[k, columns], equal_nan=True), (k, np.flatnonzero(got[t, columns] != want[k, columns]))
