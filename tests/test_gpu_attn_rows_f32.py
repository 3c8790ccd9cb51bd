"""Attention of many rows with Float32 operands on the matrix cores (csrc/attn_rows.hip) against 64 bits, at the
edges of its tiles (32 queries, 32 keys, heads of 64 and 128 and sizes between), through every entry point that
reaches it.

Bound: operands are off by 2^-24 of themselves at most, scores, softmax and sums are Float32 as in the row kernel the suite holds to
2e-5 elsewhere; 2e-6 of a row's norm is four times what is seen."""
import numpy as np
import pytest

from litenn_amd.formats import DT_F16, DT_F32

pytestmark = pytest.mark.gpu


def plain(q, k, v, scale, first, window=None, sinks=None, softcap=0.0, mask=None, slopes=None, causal=True):
    m, heads, dim = q.shape
    share = heads // k.shape[1]
    out = np.zeros((m, heads, v.shape[2]))
    for h in range(heads):
        s = q[:, h] @ k[:, h // share].T * scale
        if softcap:
            s = softcap * np.tanh(s / softcap)
        if mask is not None:
            s = s + mask * slopes[h]
        i, j = first + np.arange(m)[:, None], np.arange(k.shape[0])[None, :]
        hidden = (j > i if causal else np.zeros_like(i * j, bool)) | (i - j >= (window or 1 << 40))
        s = np.where(hidden, -np.inf, s)
        top = s.max(axis=1, keepdims=True)
        if sinks is not None:
            top = np.maximum(top, sinks[h])
        e = np.exp(s - top)
        total = e.sum(axis=1, keepdims=True) + (np.exp(sinks[h] - top) if sinks is not None else 0.0)
        out[:, h] = e / total @ v[:, h // share]
    return out.reshape(m, -1)


def inputs(seed, m, keys, heads, kv, dim, dtype, spread=1.0):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((m, heads, dim)).astype(np.float32) * np.float32(spread)
    k, v = (rng.standard_normal((keys, kv, dim)).astype(np.float32) for _ in range(2))
    if dtype == DT_F16:
        k, v = k.astype(np.float16), v.astype(np.float16)
    return q, k, v


def worst(got, want):
    return (np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)).max()


CASES = [(16, 96, 3, 3, 128), (31, 129, 8, 2, 128), (32, 97, 4, 1, 64), (33, 128, 8, 8, 128), (65, 160, 2, 1, 64), (100, 333, 16, 4, 128),
         (40, 200, 2, 2, 72), (17, 500, 5, 5, 8), (16, 511, 3, 3, 128), (35, 529, 4, 2, 128), (16, 800, 3, 1, 64), (40, 512, 129, 43, 8),
         # four and eight groups on either side of 256 workgroups, Float32 tiles of a wavefront's own and in pairs
         (101, 417, 16, 4, 128), (65, 1003, 32, 8, 128), (290, 290, 16, 16, 128), (290, 1001, 32, 8, 128), (97, 130, 96, 96, 120),
         (290, 291, 32, 8, 128), (350, 352, 24, 8, 64)]


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("m,keys,heads,kv,dim", CASES)
def test_causal_rows(hip, dtype, m, keys, heads, kv, dim):
    q, k, v = inputs(1, m, keys, heads, kv, dim, dtype, spread=3.0)
    q[0] *= np.float32(1e-12)  # every query keeps its own scale
    T = hip.Tensor.from_numpy
    got = hip.attn_rows(T(q), T(k), T(v), m, keys - m, heads, kv, dim, precise=True).numpy()
    want = plain(*(a.astype(np.float64) for a in (q, k, v)), dim ** -0.5, keys - m)
    assert worst(got, want) <= 2e-6


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("m,keys,heads,kv,dim", [(16, 96, 6, 3, 128), (37, 130, 8, 8, 64), (33, 545, 8, 4, 128), (20, 2050, 2, 2, 64),
                                                   (4, 128, 2, 1, 120), (5, 1029, 3, 1, 128), (32, 75, 24, 8, 64),
                                                   (130, 137, 64, 8, 128)])
@pytest.mark.parametrize("causal", [True, False])
def test_options(hip, dtype, m, keys, heads, kv, dim, causal):
    q, k, v = inputs(2, m, keys, heads, kv, dim, dtype)
    rng = np.random.default_rng(3)
    mask = -np.abs(rng.standard_normal((m, keys))).astype(np.float32) * 4
    mask[:, 40:70] = -np.inf                       # whole tiles of hidden keys
    mask[3] = np.where(np.arange(keys) == 5, 0.0, np.finfo(np.float32).min)  # the type's lowest value
    sinks = rng.standard_normal(heads).astype(np.float32)
    power = 2 ** int(np.log2(heads))
    slopes = [2.0 ** (-8.0 / power * (h + 1)) if h < power else 2.0 ** (-4.0 / power * (2 * (h - power) + 1)) for h in range(heads)]
    T = hip.Tensor.from_numpy
    got = hip.flash_attn_ext(T(q), T(k), T(v), m, keys, heads, kv, dim, scale=dim ** -0.5, max_bias=8.0, logit_softcap=20.0, mask=T(mask),
                             sinks=T(sinks), causal=causal, query_position_offset=keys - m).numpy()
    want = plain(*(a.astype(np.float64) for a in (q, k, v)), dim ** -0.5, keys - m, sinks=sinks, softcap=20.0,
                 mask=mask.astype(np.float64), slopes=slopes, causal=causal)
    assert worst(got, want) <= 2e-6


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("m,keys,heads,kv,dim", [(4, 79, 8, 8, 72), (4, 80, 8, 4, 80), (1, 130, 32, 8, 112), (4, 799, 4, 2, 104), (4, 800, 4, 2, 104),
                                                   (8, 111, 64, 8, 96), (15, 299, 36, 4, 88), (15, 300, 36, 4, 88), (16, 96, 4, 4, 80), (12, 64, 128, 8, 96)])
@pytest.mark.parametrize("softcap", [0.0, 30.0])
def test_options_of_few_rows(hip, dtype, m, keys, heads, kv, dim, softcap):
    """Heads between 64 and 128, on either side of where the tiles begin."""
    q, k, v = inputs(4, m, keys, heads, kv, dim, dtype)
    rng = np.random.default_rng(5)
    mask = -np.abs(rng.standard_normal((m, keys))).astype(np.float32)
    mask[:, :20] = -np.inf
    sinks = rng.standard_normal(heads).astype(np.float32)
    T = hip.Tensor.from_numpy
    got = hip.flash_attn_ext(T(q), T(k), T(v), m, keys, heads, kv, dim, scale=dim ** -0.5, logit_softcap=softcap, mask=T(mask),
                             sinks=T(sinks), causal=True, query_position_offset=keys - m).numpy()
    want = plain(*(a.astype(np.float64) for a in (q, k, v)), dim ** -0.5, keys - m, sinks=sinks, softcap=softcap,
                 mask=mask.astype(np.float64), slopes=[1.0] * heads)
    assert worst(got, want) <= 2e-6


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("m", [7, 40])
def test_scores_that_saturate_the_soft_cap(hip, dtype, m):
    """Capped scores of 43.7 to 44.3, where exp(2x) comes to the end of its range, beside small ones: tanh is 1, on
    either side of the number of rows from which the matrix cores are used."""
    keys, heads, dim, cap = 128, 2, 64, 20.0
    rng = np.random.default_rng(6)
    k = np.zeros((keys, 1, dim), np.float32)
    k[:, 0, 0] = np.where(np.arange(keys) % 3 == 0, np.linspace(43.7, 44.3, keys), rng.uniform(0.9, 1.1, keys)).astype(np.float16)
    k[0::2, 0, 0] *= -1
    v = rng.standard_normal((keys, 1, dim)).astype(np.float32)
    if dtype == DT_F16:
        k, v = k.astype(np.float16), v.astype(np.float16)
    q = np.zeros((m, heads, dim), np.float32)
    q[:, :, 0] = cap
    T = hip.Tensor.from_numpy
    got = hip.flash_attn_ext(T(q), T(k), T(v), m, keys, heads, 1, dim, scale=1.0, logit_softcap=cap, causal=False).numpy()
    assert worst(got, plain(*(a.astype(np.float64) for a in (q, k, v)), 1.0, 0, softcap=cap, causal=False)) <= 2e-6


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("m", [1, 7, 40])
def test_a_mask_that_hides_the_first_keys(hip, dtype, m):
    keys, heads, dim = 130, 2, 64
    q, k, v = inputs(8, m, keys, heads, 1, dim, dtype)
    mask = np.zeros((m, keys), np.float32)
    mask[:, :37] = -np.inf
    T = hip.Tensor.from_numpy
    got = hip.flash_attn_ext(T(q), T(k), T(v), m, keys, heads, 1, dim, scale=dim ** -0.5, mask=T(mask), causal=False).numpy()
    want = plain(*(a.astype(np.float64) for a in (q, k, v)), dim ** -0.5, 0, mask=mask.astype(np.float64), slopes=[1.0] * heads, causal=False)
    assert worst(got, want) <= 2e-6


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("dim", [64, 128])
def test_operands_far_below_their_rows_largest(hip, dtype, dim):
    """A query's small elements beside one 2^26 times as large that meets zeros, and values of keys whose weights are
    2^-30 and 2^-36 of the largest: each counts with its own 24 bits."""
    m, keys, heads = 40, 200, 2
    q, k, v = inputs(7, m, keys, heads, 1, dim, DT_F32)
    q[:, :, 5] = np.float32(2.0 ** 26)
    k[:, :, 5] = 0.0
    k, v = k.astype(np.float16), v.astype(np.float16)
    T = hip.Tensor.from_numpy

    def error(q, k, v):
        k, v = (a.astype(np.float16 if dtype == DT_F16 else np.float32) for a in (k, v))
        got = hip.attn_rows(T(q), T(k), T(v), m, keys - m, heads, 1, dim, precise=True).numpy()
        return worst(got, plain(*(a.astype(np.float64) for a in (q, k, v)), dim ** -0.5, keys - m))
    assert error(q, k, v) <= 2e-6
    q[:], k[:] = 0.0, 0.0
    q[:, :, 0] = np.sqrt(dim)
    k[1:, 0, 0] = np.where(np.arange(keys - 1) % 2, -30 * np.log(2.0), -36 * np.log(2.0))
    v[0], v[1:] = 1e-4 * v[0], 3e4 * np.sign(v[1:])
    assert error(q, k, v) <= 2e-6


@pytest.mark.parametrize("m,keys,heads,dim,vdim,window,at", [(16, 100, 3, 24, 40, 96, 84), (50, 150, 2, 128, 64, 97, 100), (96, 96, 4, 128, 128, 200, 0),
                                                                 (40, 95, 3, 80, 80, 200, 55), (40, 90, 35, 80, 80, 70, 50), (17, 65, 2, 64, 64, 65, 48)])
def test_float32_windows(hip, m, keys, heads, dim, vdim, window, at):
    rng = np.random.default_rng(4)
    q = rng.standard_normal((m, heads, dim)).astype(np.float32)
    kv = rng.standard_normal((keys, heads * (dim + vdim))).astype(np.float32)
    sinks, gate = rng.standard_normal(heads).astype(np.float32), rng.standard_normal((m, heads * vdim)).astype(np.float32)
    T = hip.Tensor.from_numpy
    got = hip.window_attn(T(q), T(kv), m, keys, heads, dim, vdim, window, scale=0.2, key_position=7, query_position=7 + at, sinks=T(sinks),
                          gate=T(gate)).numpy()
    k, v = kv[:, :heads * dim].reshape(keys, heads, dim), kv[:, heads * dim:].reshape(keys, heads, vdim)
    want = plain(*(a.astype(np.float64) for a in (q, k, v)), 0.2, at, window, sinks) / (1.0 + np.exp(-gate.astype(np.float64)))
    assert worst(got, want) <= 2e-6


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
def test_a_value_that_is_not_finite_stays_with_the_queries_that_see_it(hip, dtype):
    m, keys, heads, dim = 40, 140, 2, 128
    q, k, v = inputs(5, m, keys, heads, 1, dim, dtype)
    T = hip.Tensor.from_numpy
    clean = hip.attn_rows(T(q), T(k), T(v), m, keys - m, heads, 1, dim, precise=True).numpy()
    bad = v.copy()
    bad[keys - 10, 0, 3], bad[keys - 5, 0, 90] = np.inf, np.nan
    got = hip.attn_rows(T(q), T(k), T(bad), m, keys - m, heads, 1, dim, precise=True).numpy().reshape(m, heads, dim)
    clean = clean.reshape(m, heads, dim)
    # (a query whose tile held the value is computed again in another order)
    assert worst(got[:m - 10].reshape(m - 10, -1), clean[:m - 10].reshape(m - 10, -1)) <= 2e-6
    assert np.all(got[m - 10:, :, 3] == np.inf) and np.all(np.isnan(got[m - 5:, :, 90]))
    rest = np.delete(got, [3, 90], axis=2), np.delete(clean, [3, 90], axis=2)
    assert np.linalg.norm(rest[0] - rest[1]) <= 2e-6 * np.linalg.norm(rest[1])


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("spread", [0.02, 0.32, 0.345, 0.355, 1.0, 8.0])
@pytest.mark.parametrize("m,keys", [(33, 129), (64, 96), (40, 700)])
def test_soft_caps_on_both_sides_of_the_series(hip, dtype, spread, m, keys):
    """The largest score is `spread` of the cap: the series' tiles alone, both kinds and the layer's form alone; key tiles that
    all queries see whole, and the ones where the first and the last key of a tile is the first that one does not."""
    heads, dim, cap = 3, 64, 7.0
    q, k, v = inputs(5, m, keys, heads, 1, dim, dtype)
    s = np.abs(np.einsum("ihd,jd->hij", q.astype(np.float64), k[:, 0].astype(np.float64))).max()
    q *= np.float32(spread * cap / s)
    T = hip.Tensor.from_numpy
    got = hip.flash_attn_ext(T(q), T(k), T(v), m, keys, heads, 1, dim, scale=1.0, logit_softcap=cap,
                             causal=True, query_position_offset=keys - m).numpy()
    assert worst(got, plain(*(a.astype(np.float64) for a in (q, k, v)), 1.0, keys - m, softcap=cap)) <= 4e-6


@pytest.mark.parametrize("dtype", [DT_F16, DT_F32])
@pytest.mark.parametrize("m,keys", [(33, 129), (64, 64), (40, 700)])
def test_soft_caps_of_a_query_hang_on_its_own_scores_alone(hip, dtype, m, keys):
    """Keys that the first rows do not see, and the other queries, grow beyond the series' range: the first rows keep their bits."""
    heads, dim, seen = 3, 64, m // 3
    q, k, v = inputs(6, m, keys, heads, 1, dim, dtype)
    T = hip.Tensor.from_numpy

    def run(q, k):
        got = hip.flash_attn_ext(T(q), T(k), T(v), m, keys, heads, 1, dim, scale=0.01, logit_softcap=7.0, causal=True,
                                 query_position_offset=keys - m).numpy()
        return got[:seen]
    hidden, others = k.copy(), q.copy()
    hidden[keys - m + seen:] *= 16
    others[seen:] *= 300
    want = run(q, k)
    assert np.array_equal(run(q, hidden), want) and np.array_equal(run(others, k), want)
