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
