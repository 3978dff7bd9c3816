"""Weights that are all bf16 numbers against the same with one in each matrix that is none, by its last bit: the products of
the former leave out the partial products whose factor is zero, the others take all of them.  What a checkpoint stores
them in makes no difference."""
import json

import numpy as np
import pytest

import tutilorn_model as tm
import zabutar_model as zm
import zabutar_oracle as zo
from test_safetensors_host import write_safetensors

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import shainet_amd as sa

    assert sa.HIP.fully_available(), "no gfx950 device or libshainet_hip_kernels.so missing"
    return sa


def bf16(a):
    """The values cut to what a bf16 holds."""
    return (np.ascontiguousarray(a, np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)


def write(folder, cfg, weights, stored_bf16, nudge=True):
    folder.mkdir()
    (folder / "config.json").write_text(json.dumps(cfg))
    out = {}
    for name, a in weights.items():
        a = np.array(a, np.float32)
        short = stored_bf16(name)
        if not short and a.ndim == 2 and nudge:
            a.reshape(-1).view(np.uint32)[a.size // 2] ^= 1
        raw = (a.view(np.uint32) >> 16).astype("<u2") if short else a
        out[name] = ("BF16" if short else "F32", np.shape(weights[name]), raw.tobytes())
    write_safetensors(folder / "model.safetensors", out)
    return str(folder)


def llama(d, ff, seed, vocab=260):
    H, KV, hd = 2, 1, 32
    cfg = {"model_type": "llama", "vocab_size": vocab, "hidden_size": d, "num_attention_heads": H, "num_hidden_layers": 1,
           "intermediate_size": ff, "num_key_value_heads": KV, "head_dim": hd, "tie_word_embeddings": False, "rms_norm_eps": 1e-6}
    r = np.random.default_rng(seed)

    def matrix(o, i):
        return bf16(r.standard_normal((o, i), np.float32) * np.float32(i ** -0.5))

    p = "model.layers.0."
    w = {"model.embed_tokens.weight": bf16(r.standard_normal((vocab, d), np.float32)), "lm_head.weight": matrix(vocab, d),
         p + "self_attn.q_proj.weight": matrix(H * hd, d), p + "self_attn.k_proj.weight": matrix(KV * hd, d),
         p + "self_attn.v_proj.weight": matrix(KV * hd, d), p + "self_attn.o_proj.weight": matrix(d, H * hd),
         p + "mlp.gate_proj.weight": matrix(ff, d), p + "mlp.up_proj.weight": matrix(ff, d), p + "mlp.down_proj.weight": matrix(d, ff)}
    for name in ("model.norm", p + "input_layernorm", p + "post_attention_layernorm"):
        w[name + ".weight"] = bf16(1 + 0.1 * r.standard_normal(d, np.float32))
    return cfg, w


def all_logits(hip, folder, tokens):
    return hip.HFLoader.load_model(folder).run_rows(tokens, range(len(tokens))).astype(np.float64)


def assert_alike(got, want):
    """Columns of logits.  Sums of up to 8192 terms in another order: 8192^0.5 roundings of 2^-24, and as much again from
    what the products before them hand on."""
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want).all(0)
    off = np.linalg.norm(got[:, ok] - want[:, ok], axis=0) / np.linalg.norm(want[:, ok], axis=0)
    assert off.max() <= 2 * 8192 ** 0.5 * 2.0 ** -24, off.max()


# tiles of 32 rows (whole and ragged steps along K), 128 x 256 cut into pieces, shared by waiting and whole, 256 x 256 likewise
@pytest.mark.parametrize("d,ff,T", [(128, 260, 40), (132, 260, 19), (640, 2052, 100), (1024, 4096, 300), (1028, 2052, 290),
                                    (640, 4100, 1100), (1040, 8192, 2000), (1044, 8196, 2000), (1040, 4100, 3000)])
def test_bf16_weights_run_like_fp32_ones(hip, tmp_path, d, ff, T):
    cfg, w = llama(d, ff, d + T)
    w["model.norm.weight"] *= np.float32(2.0 ** 20)
    head = w["lm_head.weight"]
    head[5, 3], head[6, d - 1], head[8, 7] = np.nan, np.inf, -np.inf
    head[7] = bf16(head[7] * np.float32(2.0 ** -129))  # bf16 numbers below the normal ones among them
    tokens = np.random.default_rng(1).integers(0, cfg["vocab_size"], T)
    got = all_logits(hip, write(tmp_path / "short", cfg, w, lambda n: True), tokens)
    assert_alike(got, all_logits(hip, write(tmp_path / "long", cfg, w, lambda n: False), tokens))
    if T < 50:
        same = all_logits(hip, write(tmp_path / "same", cfg, w, lambda n: "mlp" in n, nudge=False), tokens)
        assert np.array_equal(got, same, equal_nan=True)


@pytest.mark.parametrize("long", ["k_proj", "up_proj", "down_proj", "lm_head"])
def test_one_fp32_tensor_among_bf16_ones_keeps_its_bits(hip, tmp_path, long):
    cfg, w = llama(256, 512, 3)
    r = np.random.default_rng(4)
    for name in w:
        if long in name:
            w[name] = w[name] * (1 + r.uniform(0, 2.0 ** -8, w[name].shape)).astype(np.float32)
    tokens = r.integers(0, cfg["vocab_size"], 60)
    assert_alike(all_logits(hip, write(tmp_path / "mixed", cfg, w, lambda n: long not in n), tokens),
                 all_logits(hip, write(tmp_path / "long", cfg, w, lambda n: False), tokens))


@pytest.mark.parametrize("T", [20, 400])
@pytest.mark.parametrize("long", [None, "down", "up"])
def test_other_designs_run_like_their_fp32_copies(hip, tmp_path, T, long):
    tokens = np.random.default_rng(5).integers(0, 90, T)
    for name, module, cfg in (("t", tm, tm.config([tm.layer(tm.mixer())], width=64)),
                              ("z", zm, zm.config([zm.layer(zm.hgrn2(), zm.dense()), zm.layer(zm.attention(), zm.moe())], width=64))):
        w = module.make_weights(cfg, 6)
        r = np.random.default_rng(7)
        for n in w:
            if long and n.endswith("." + long):
                w[n] = w[n] * (1 + r.uniform(0, 2.0 ** -8, np.shape(w[n]))).astype(np.float32)
        assert_alike(all_logits(hip, write(tmp_path / (name + "short"), cfg, w, lambda n: not (long and n.endswith("." + long))), tokens),
                     all_logits(hip, write(tmp_path / (name + "long"), cfg, w, lambda n: False), tokens))


@pytest.mark.parametrize("short", [True, False])
@pytest.mark.parametrize("width,ff,T", [(64, 96, 150), (60, 52, 150), (55, 47, 150), (1040, 512, 330), (1024, 516, 330), (1056, 509, 330)])
def test_experts_products_keep_every_part(hip, tmp_path, width, ff, T, short):
    """Tiles of 64 and 128 rows; lengths of K that are whole steps, pieces of four, and neither, by turns of the two products.  A
    third part of the rows left out of a product is 2e-6 to 3.5e-6 of what an expert returns, a part of the weights more; sums of
    up to 1056 terms, the norms and the activation are off by a tenth of that.  Then a last row of NaN: the rows beside it are
    fp32 sums that round every two terms, 528 times 2^-24 at random, in each of the two products."""
    cfg = zm.config([zm.layer(zm.hgrn2(heads=1, dim=4, vdim=4), zm.moe(ff=ff, experts=2, identity=0, top=1, groups=1, keep=1, shared=0))],
                    width=width)
    w = zm.make_weights(cfg, 3)
    w["l0.mix.o"] = 0 * w["l0.mix.o"]
    if not short:
        r = np.random.default_rng(7)
        for n in w:
            if ".e0." in n or ".e1." in n:
                w[n] = w[n] * (1 + r.uniform(0, 2.0 ** -8, np.shape(w[n]))).astype(np.float32)
    x = (2 * np.random.default_rng(4).standard_normal((T, width))).astype(np.float32)
    model = hip.HFLoader.load_model(write(tmp_path / "m", cfg, w, lambda n: short or ".mlp.e" not in n))
    got = model.blocks[0].forward_cached(x).astype(np.float64) - x
    with zm.watch_choices() as gaps:
        want = zo.layer(cfg, w, 0, x.astype(np.float64), {}) - x
    assert min(gaps) > 3e-6, "a choice of experts too close to call: another seed"
    assert np.linalg.norm(got - want) <= 1.2e-6 * np.linalg.norm(want), np.linalg.norm(got - want) / np.linalg.norm(want)
    kept = (T - 1) // 64 * 64  # (a chunk of the mixer, 64 rows, is not kept apart)
    x[T - 1] = np.nan
    model.clear_cache()
    got = model.blocks[0].forward_cached(x).astype(np.float64) - x
    assert np.isnan(got[T - 1]).all()
    assert np.linalg.norm(got[:kept] - want[:kept]) <= 3e-6 * np.linalg.norm(want[:kept])
