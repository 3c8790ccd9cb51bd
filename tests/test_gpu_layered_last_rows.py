"""Prompts of layered decoders whose last rows' logits alone are asked for: the last layer then makes keys, values and
states of every row, and queries, gates and what lies behind the mixer of the asked ones, one row as a step does."""
import numpy as np
import pytest

import degedra_util as du
import kulurax_util as ku
import np_degedra
import np_kulurax

pytestmark = pytest.mark.gpu

# as in the tests of whole prompts: Float32 sums of chains this long, operands rounded to bfloat16
LIMIT = {"float32": 3e-5, "bfloat16": 4e-2}

LAST = {
    "latent": (ku.config([ku.linear_attention(), ku.attention(window=70, mlp=ku.mlp())]), ku.random_weights, np_kulurax.NumpyKulurax),
    "latent_alone": (ku.config([ku.attention(heads=2, dim=136, vdim=72, kv_rank=37, q_rank=29, window=130)]), ku.random_weights, np_kulurax.NumpyKulurax),
    "linear": (ku.config([ku.attention(), ku.linear_attention(heads=3, dim=33, vdim=21, mlp=ku.mlp())], width=53), ku.random_weights,
               np_kulurax.NumpyKulurax),
    "both": (du.config([du.layer(ff=72), du.layer(ff=50)]), du.random_weights, np_degedra.NumpyDegedra),
    "both_odd": (du.config([du.layer(du.attention(3, 3, 13, 66, 1.0, 4), du.state_space(2, 35, 33, 1, 2, 3), ff=33)]), du.random_weights,
                 np_degedra.NumpyDegedra),
}


@pytest.mark.parametrize("rows", [383, 384, 401])
def test_one_row_over_cached_latents(hip, rows):
    """Both sides of the number of keys from which one asked row attends to the latents themselves."""
    cfg = ku.config([ku.linear_attention(), ku.attention(heads=5, window=390)])
    w = ku.random_weights(cfg, 21)
    toks = ku.tokens(cfg, rows, 6)
    want = np_kulurax.NumpyKulurax(cfg, ku.as_floats(w)).forward(toks)
    with hip.create_model(cfg, w, dtype="bfloat16", context_length=410) as model:
        assert ku.error(model.eval(toks, want=[rows - 1]), want[rows - 1:]) <= LIMIT["bfloat16"]


@pytest.mark.parametrize("name", ["latent", "both"])
def test_few_asked_rows_behind_whole_tiles(hip, name):
    """Float32: up to 15 rows past a tile of 64 take the tile before them too."""
    cfg, weights, plain_form = LAST[name]
    w = weights(cfg, 21)
    toks = ku.tokens(cfg, 280, 6)
    want = plain_form(cfg, ku.as_floats(w)).forward(toks)
    with hip.create_model(cfg, w, dtype="float32", context_length=300) as model:
        for past, rows, count in ((0, 130, 2), (0, 207, 15), (37, 194, 2), (37, 208, 16), (0, 143, 16), (0, 200, 9)):
            model.reset()
            if past:
                model.eval(toks[:past], want=[])
            got = model.eval(toks[past:past + rows], want=list(range(rows - count, rows)))
            assert ku.error(got, want[past + rows - count:past + rows]) <= LIMIT["float32"], (past, rows, count)
            got = model.eval(toks[past + rows:past + rows + 1])
            assert ku.error(got, want[past + rows:past + rows + 1]) <= LIMIT["float32"], (past, rows, count)


# heads and value sizes of every form of the launch that makes both mixers' outputs, at the edges of its tiles (64 queries,
# chunks of 64 tokens, two blocks of the recurrence to a workgroup), few workgroups and many, four taps and others
PAIRS = {
    "64_64": du.layer(du.attention(4, 2, 64, 70, 0.1, 32), du.state_space(3, 64, 128, 1, 1, 4)),
    "64_odd": du.layer(du.attention(3, 3, 40, 21, 0.2, 40), du.state_space(4, 36, 33, 1, 2, 4)),
    "128": du.layer(du.attention(8, 2, 128, 100, 0.1, 128), du.state_space(2, 70, 65, 2, 1, 4)),
    "96": du.layer(du.attention(5, 5, 96, 40, 0.1, 64), du.state_space(1, 20, 20, 1, 1, 4)),
    "three_taps": du.layer(du.attention(4, 2, 64, 70, 0.1, 32), du.state_space(4, 32, 64, 2, 2, 3)),
    "beyond": du.layer(du.attention(2, 2, 136, 70, 0.1, 100), du.state_space(2, 32, 64, 1, 1, 4)),
    "many": du.layer(du.attention(64, 8, 64, 200, 0.1, 32), du.state_space(32, 64, 64, 2, 2, 4)),
}


@pytest.mark.parametrize("dtype", sorted(LIMIT))
@pytest.mark.parametrize("name", sorted(PAIRS))
def test_both_mixers_in_one_launch(hip, name, dtype):
    cfg = du.config([PAIRS[name]])
    w = du.random_weights(cfg, 8)
    plain = np_degedra.NumpyDegedra(cfg, du.as_floats(w))
    toks = ku.tokens(cfg, 330, 6)
    want = plain.forward(toks)
    with hip.create_model(cfg, w, dtype=dtype, context_length=330) as model:
        for rows in (4, 63, 64, 65, 128, 330):
            model.reset()
            assert ku.error(model.eval(toks[:rows]), want[:rows]) <= LIMIT[dtype], rows


@pytest.mark.parametrize("dtype", sorted(LIMIT))
@pytest.mark.parametrize("name", sorted(LAST))
def test_rows_asked_for(hip, name, dtype):
    """Sizes around the tiles of queries and chunks of tokens, behind a first portion, one row and several; the step behind
    the prompt reads all that it kept."""
    cfg, weights, plain_form = LAST[name]
    w = weights(cfg, 21)
    plain = plain_form(cfg, ku.as_floats(w))
    toks = ku.tokens(cfg, 280, 6)
    want = plain.forward(toks)
    with hip.create_model(cfg, w, dtype=dtype, context_length=300) as model:
        for past in (0, 37):
            for rows in (4, 15, 16, 63, 64, 65, 129, 200):
                for count in (1, 2, 64):
                    if count > rows:
                        continue
                    model.reset()
                    if past:
                        model.eval(toks[:past], want=[])
                    got = model.eval(toks[past:past + rows], want=list(range(rows - count, rows)))
                    end = past + rows
                    assert ku.error(got, want[end - count:end]) <= LIMIT[dtype], (past, rows, count)
                    got = model.eval(toks[end:end + 1])
                    assert ku.error(got, want[end:end + 1]) <= LIMIT[dtype], (past, rows, count)
