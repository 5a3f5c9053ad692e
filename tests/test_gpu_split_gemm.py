"""Projections on split operands (F16 matrix cores, three products) at the
shapes where the kernel's tiles can go wrong: single 32-k blocks, slices of one
to eight blocks, rows and columns that end inside a small or a large tile,
narrow widths, both tile orders, and every epilogue of the text path, against
the scalar oracle; operands whose channels spread far apart; and attention on
split head rows."""
import numpy as np
import pytest

import svl_amd
import svl_synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def small_config(hidden, inter, ple, heads, kv, hd, out):
    c = svl_synth.config_a(2, 97)
    c.update(hidden_size=hidden, intermediate_size=inter, hidden_size_per_layer_input=ple,
             num_attention_heads=heads, num_key_value_heads=kv, head_dim=hd, embedding_dim=out,
             sliding_window=16)
    return c


# hidden, FFN, PLE, heads, KV heads, head dim, embedding width: K of 32, 64, 96, 128, 160 and 256;
# outputs of 40 and 33 columns (runs that end inside a vector store), generic and MFMA attention
SHAPES = [(32, 32, 32, 2, 1, 16, 40), (64, 96, 32, 2, 1, 32, 33), (128, 160, 64, 2, 2, 64, 128),
          (256, 512, 128, 3, 1, 64, 256), (96, 128, 96, 1, 1, 128, 100)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_split_projections_match_the_oracle(shape):
    cfg = small_config(*shape)
    w = svl_synth.weights(cfg, seed=3)
    model = svl_amd.TextModel(svl_amd.TextConfig.from_json_value(cfg), w)
    oracle = O.OracleTextModel(cfg, w)
    # one row, a row that ends inside a 16-row block, one past a 32- and a 64-row tile
    rows = svl_synth.token_rows(97, [1, 17, 33, 65], seed=4)
    outs = model.forward_batch(rows, capture_hidden=True)
    for row, out in zip(rows, outs):
        ref = oracle.forward(row)
        # float32 sums of at most 512 terms through two layers: the oracle bound of the model tests
        assert np.abs(out.normalized() - ref["normalized"]).max() <= 1e-4
        assert np.abs(out.projected() - ref["projected"]).max() <= 1e-4 * max(
            1.0, float(np.abs(ref["projected"]).max()))
        alone = model.forward(row)
        assert np.array_equal(alone.normalized(), out.normalized())
    model.close()


# tokens and embedding width: outputs that end inside a large tile and inside a run of four
# columns, in the plain order (100 and 803 columns) and the grouped one (1301 and 2307); 64x64
# tiles, then 64x128 and 128x128 ones by turns
@pytest.mark.parametrize("tokens,out", [(24000, 100), (27000, 100), (24000, 803), (12000, 803),
                                        (15700, 1301), (12000, 1301), (9000, 2307)])
def test_large_tiles_end_inside_the_output(tokens, out):
    cfg = small_config(64, 64, 32, 1, 1, 32, out)
    w = svl_synth.weights(cfg, seed=15)
    model = svl_amd.TextModel(svl_amd.TextConfig.from_json_value(cfg), w)
    n = 61
    lengths = [n] * (tokens // n) + [tokens % n or 1]
    rows = svl_synth.token_rows(97, lengths, seed=16)
    outs = model.forward_batch(rows)
    oracle = O.OracleTextModel(cfg, w)
    for i in (0, len(rows) // 2, len(rows) - 2, len(rows) - 1):
        alone = model.forward(rows[i])  # small tiles
        assert np.array_equal(alone.projected(), outs[i].projected())
        ref = oracle.forward(rows[i])["projected"]
        # as in test_split_projections_match_the_oracle
        assert np.abs(outs[i].projected() - ref).max() <= 1e-4 * max(1.0, float(np.abs(ref).max()))
    model.close()


@pytest.mark.parametrize("gain", [2.0 ** -60, 2.0 ** 20, 3e-3])
def test_split_scales_follow_the_weights(gain):
    """Norm weights and projections far from one: the operands' power-of-two scales keep the
    products exact to float32 rounding (the gains cancel in the next norm; squares of
    the activations have to stay below 2^128)."""
    cfg = small_config(64, 96, 32, 2, 1, 32, 64)
    w = svl_synth.weights(cfg, seed=5)
    w = {k: (v * np.float32(gain) if k.endswith(("pre_feedforward_layernorm.weight",
                                                 "o_proj.weight")) else v) for k, v in w.items()}
    model = svl_amd.TextModel(svl_amd.TextConfig.from_json_value(cfg), w)
    row = svl_synth.token_rows(97, [29], seed=6)[0]
    ref = O.OracleTextModel(cfg, w).forward(row)["normalized"]
    assert np.abs(model.forward(row).normalized() - ref).max() <= 1e-4
    model.close()


# head_dim 256, 512 (shape B's global layers) and 64, one and two layers deep: the rows alone take
# the short-grid variants (several waves per 16 queries), the whole batch the large-grid ones
@pytest.mark.parametrize("heads,kv,hd", [(3, 1, 256), (4, 2, 256), (4, 1, 512), (4, 4, 64)])
def test_split_attention_matches_the_oracle_and_itself(heads, kv, hd):
    cfg = small_config(256, 128, 64, heads, kv, hd, 128)
    cfg.update(sliding_window=40)
    w = svl_synth.weights(cfg, seed=7)
    model = svl_amd.TextModel(svl_amd.TextConfig.from_json_value(cfg), w)
    oracle = O.OracleTextModel(cfg, w)
    # below one key tile, at its edges, past the window, and one long row
    lengths = [1, 31, 32, 33, 64, 65, 129, 300] + [257] * 28
    rows = svl_synth.token_rows(97, lengths, seed=8)
    outs = model.forward_batch(rows)
    for i in range(8):
        alone = model.forward(rows[i])
        assert np.array_equal(alone.projected(), outs[i].projected())
        assert np.abs(alone.normalized() - oracle.forward(rows[i])["normalized"]).max() <= 1e-4
    model.close()


def cancelling_gains(w, layers, heads_group, rng, k):
    """The same function with some channels 2^k stronger where they are written and 2^-k weaker
    where they are read: norm outputs, GeGLU and PLE activations, query and key pairs."""
    w = dict(w)
    up = np.float32(2.0 ** k)

    def scaled(name, index, gain):
        w[name] = w[name].copy()
        w[name][index] *= gain

    def channel(norm, readers):
        c = int(rng.integers(len(w[norm])))
        scaled(norm, c, up)
        for r in readers:
            scaled(r, (slice(None), c), 1 / up)

    pre = "language_model."
    channel(pre + "norm.weight", [pre + "embedding_projection.weight"])
    ps = [f"{pre}layers.{l}." for l in range(layers)]
    channel(pre + "ple.per_layer_projection_norm.weight",
            [p + "ple_block.per_layer_projection.weight" for p in ps])
    for p in ps:
        channel(p + "input_layernorm.weight", [f"{p}self_attn.{x}_proj.weight" for x in "qkv"])
        channel(p + "pre_feedforward_layernorm.weight",
                [p + "mlp.gate_proj.weight", p + "mlp.up_proj.weight"])
        j = int(rng.integers(len(w[p + "mlp.up_proj.weight"])))
        scaled(p + "mlp.up_proj.weight", j, up)
        scaled(p + "mlp.down_proj.weight", (slice(None), j), 1 / up)
        i = int(rng.integers(heads_group // 2))
        pair = [i, i + heads_group // 2]
        scaled(p + "self_attn.q_norm.weight", pair, up)
        scaled(p + "self_attn.k_norm.weight", pair, 1 / up)
    return w


@pytest.mark.parametrize("heads,kv,hd", [(2, 1, 64), (3, 1, 256), (2, 1, 512), (2, 1, 128)])
@pytest.mark.parametrize("k", [20, 7, -17])
def test_channel_gains_that_cancel_leave_the_bits(heads, kv, hd, k):
    """Every channel of a split operand has a scale of its own: one that stands out by any power of
    two, undone by the weight that reads it, changes no bit (one scale per tensor held the other
    channels in 2^k fewer)."""
    cfg = small_config(128, 160, 64, heads, kv, hd, 96)
    w = svl_synth.weights(cfg, seed=9)
    tc = svl_amd.TextConfig.from_json_value(cfg)
    rows = svl_synth.token_rows(97, [5, 40], seed=10)
    outs = []
    for v in (w, cancelling_gains(w, 2, hd, np.random.default_rng(k + 100), k)):
        model = svl_amd.TextModel(tc, v)
        outs.append([r.projected() for r in model.forward_batch(rows)])
        model.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_strong_gate_and_up_channels_match_the_oracle():
    """A few gate and up rows 2^8 stronger (products of 2^16), not undone anywhere."""
    cfg = small_config(128, 160, 64, 2, 1, 64, 96)
    w = svl_synth.weights(cfg, seed=11)
    for l in range(2):
        for name in ("gate_proj", "up_proj"):
            w[f"language_model.layers.{l}.mlp.{name}.weight"][[3, 77]] *= np.float32(256.0)
    model = svl_amd.TextModel(svl_amd.TextConfig.from_json_value(cfg), w)
    row = svl_synth.token_rows(97, [29], seed=12)[0]
    ref = O.OracleTextModel(cfg, w).forward(row)["normalized"]
    # two layers of float32 sums of at most 160 terms: a few 2^-23 of the vector's norm 1
    assert np.abs(model.forward(row).normalized() - ref).max() <= 4e-6
    model.close()


@pytest.mark.parametrize("where", ["norm", "key pair"])
def test_silent_outliers_keep_the_other_channels(where):
    """An outlier that no later weight undoes and whose values happen to be zero: a norm weight of
    2^30 over a column of zeros (its bound leaves the others' columns 2^30 below it, so the model
    runs on FP32 operands), and query weights of 2^24 on a pair whose key weights are zero. In
    FP32 neither changes anything."""
    cfg = small_config(128, 160, 64, 2, 1, 64, 96)
    w = svl_synth.weights(cfg, seed=13)
    p = "language_model.layers.0."
    if where == "norm":
        w["language_model.embed_tokens.weight"][:, 17] = 0.0
    else:
        w[p + "self_attn.k_norm.weight"][[4, 36]] = 0.0
    row = svl_synth.token_rows(97, [23], seed=14)[0]
    ref = O.OracleTextModel(cfg, w).forward(row)["normalized"]
    if where == "norm":
        w[p + "input_layernorm.weight"][17] *= np.float32(2.0 ** 30)
    else:
        w[p + "self_attn.q_norm.weight"][[4, 36]] *= np.float32(2.0 ** 24)
    model = svl_amd.TextModel(svl_amd.TextConfig.from_json_value(cfg), w)
    assert np.abs(model.forward(row).normalized() - ref).max() <= 4e-6  # as above
    model.close()
