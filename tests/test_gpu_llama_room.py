"""What a LLaMA model holds of the card's memory for products with Float32 operands: sums of ranges of K for the rows that a
matrix meets, which for the head are those whose logits are asked for."""
import ctypes as C

import numpy as np
import pytest

from litenn_amd import hiprt, synth
from litenn_amd.formats import Q4_0, Q6_K

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    hiprt._check(hiprt.rt().hipMemGetInfo(C.byref(free), C.byref(total)))
    return free.value


def test_the_head_has_room_for_the_rows_that_it_meets(hip):
    """300 tokens, a Q6_K head of 40000 rows: 96 MB of sums where all logits are asked for, none for one row of them."""
    rows, vocab, d = 300, 40000, 4096
    cfg = synth.LLaMAConfig("t", 1, d, 32, 8, 512, vocab, 320, formats={"default": Q4_0, "output": Q6_K})
    model = hip.LLaMA.from_config(cfg)
    model.load(synth.llama_tensors(cfg, 3))
    toks = np.random.default_rng(5).integers(0, vocab, rows).astype(np.int32)
    model.eval(toks[:8], all_logits=False)  # the code is on the card
    model.reset()
    before = free_bytes()
    one = model.eval(toks, all_logits=False)
    held = before - free_bytes()
    assert held < 60e6, held
    model.reset()
    whole = model.eval(toks)
    assert before - free_bytes() - held > 90e6
    # the last row's query and what follows the last block's keys meet operands in 32 bits either way, in other orders
    assert np.linalg.norm(whole[-1] - one) <= 1e-4 * np.linalg.norm(one)
    model.reset()
    some = model.eval(toks[:70])
    assert np.linalg.norm(some - whole[:70]) <= 1e-4 * np.linalg.norm(some)
    model.close()
