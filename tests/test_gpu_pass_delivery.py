"""How a pass's ids reach the device and its results the host: runs of more ids than the pinned memory has room for,
passes of one run, states of all layers cleared by one call, results read at once by several threads."""
import os
import threading

import numpy as np
import pytest

import degedra_util as du
import kulurax_util as ku

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [65536, 65537, 65900])
def test_runs_longer_than_the_pinned_ids(hip, rows):
    """The same passes, whether their ids come out of pinned memory (65536 of a run) or are copied."""
    cfg = ku.config([ku.linear_attention(), ku.attention(window=5)], width=16)
    toks = ku.tokens(cfg, rows, 3)
    with hip.create_model(cfg, ku.random_weights(cfg, 4), dtype="float32", context_length=rows + 2) as model:
        whole = model.eval(toks, want=[0, rows - 2, rows - 1])
        step = model.eval(toks[:1])
        model.reset()
        first = model.eval(toks[:4096 * 9], want=[0])
        rest = model.eval(toks[4096 * 9:], want=[rows - 4096 * 9 - 2, rows - 4096 * 9 - 1])
        assert np.array_equal(whole, np.concatenate([first, rest]))
        assert np.array_equal(step, model.eval(toks[:1]))


def test_reset_clears_every_layer(hip):
    cfg = du.config([du.layer(ff=40), du.layer(du.attention(3, 3, 13, 6, 1.0, 4), du.state_space(2, 35, 33, 1, 2, 3)), du.layer(ff=24)])
    toks = ku.tokens(cfg, 90, 3)
    w = du.random_weights(cfg, 4)
    with hip.create_model(cfg, w, dtype="float32", context_length=100) as model:
        want = [model.eval(toks[:80]), model.eval(toks[80:81])]
        for _ in range(3):
            model.reset()
            assert np.array_equal(model.eval(toks[:80]), want[0])
            assert np.array_equal(model.eval(toks[80:81]), want[1])


def eval_in_threads(hip, count):
    cfg = ku.config([ku.linear_attention(mlp=ku.mlp()), ku.attention()])
    toks = ku.tokens(cfg, 60, 3)
    models = [hip.create_model(cfg, ku.random_weights(cfg, seed), dtype="float32", context_length=64) for seed in range(count)]
    want = [np.concatenate([m.eval(toks[:20], want=[19])] + [m.eval(toks[i:i + 1]) for i in range(20, 60)]) for m in models]
    wrong = []

    def steps(m, expected):
        for _ in range(5):
            m.reset()
            got = np.concatenate([m.eval(toks[:20], want=[19])] + [m.eval(toks[i:i + 1]) for i in range(20, 60)])
            if not np.array_equal(got, expected):
                wrong.append(m)

    threads = [threading.Thread(target=steps, args=p) for p in zip(models, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m in models:
        m.close()
    assert not wrong


def test_models_in_threads(hip):
    eval_in_threads(hip, 3)


def test_models_in_more_threads_than_cores(hip):
    """Threads that look at the marks of their passes while others, on the same core, have launches to make."""
    cores = os.sched_getaffinity(0)
    os.sched_setaffinity(0, sorted(cores)[:1])  # of this thread, and those that it starts
    try:
        eval_in_threads(hip, 8)
    finally:
        os.sched_setaffinity(0, cores)
