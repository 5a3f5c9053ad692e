"""Projections on split operands (F16 matrix cores, three products) at the
shapes where the kernel's tiles can go wrong: single 32-k blocks, slices of one
to eight blocks, rows and columns that end inside a tile, narrow widths, and
every epilogue of the text path, against the scalar oracle."""
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
