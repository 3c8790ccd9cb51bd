"""The quantised matmul of several rows with Float32 operands (integer weights times split activations on the
matrix cores) against the numpy decoder and a product in 64 bits.  Sizes lie at the edges of its tiles (32 rows of
either side, 256 elements of K) and on both sides of every rule that picks a form.

Bound: a weight is exact, an activation keeps 22 bits and more (relative error 2^-23 at most), and Float32 sums of
k random products of like size err by about sqrt(log2 k) 2^-24 of |x| |W| / sqrt(k), the size such a sum has (a single
output may happen to cancel to less, which no summation order can follow); 1e-6 is four times what is seen."""
import numpy as np
import pytest

import np_decoders
from litenn_amd import synth
from litenn_amd.formats import Q4_0, Q4_K, Q5_K, Q6_K, Q8_0
from litenn_amd.llama import MATMUL_PRECISE

pytestmark = pytest.mark.gpu
FORMATS = [Q4_0, Q8_0, Q4_K, Q5_K, Q6_K]


def errors(hip, fmt, m, n, k, residual=False):
    wq = synth.model_weights(fmt, n, k, 21, m, n)
    x = synth.activations(m, k, 22, m)
    x[m // 2] *= np.float32(1e-20)  # every row keeps its own scale
    res = synth.activations(m, n, 23, 1) if residual else None
    got = hip.mul_mat_q(fmt, hip.Tensor.from_numpy(wq), n, k, hip.Tensor.from_numpy(x),
                        residual=hip.Tensor.from_numpy(res) if residual else None, flags=MATMUL_PRECISE).numpy()
    w = np_decoders.decode(fmt, wq, k).astype(np.float64)
    want = x.astype(np.float64) @ w.T
    size = np.linalg.norm(x.astype(np.float64), axis=1) * np.linalg.norm(w) / np.sqrt(k)
    if residual:
        want += res
        size = np.hypot(size, np.linalg.norm(res, axis=1))
    return np.linalg.norm(got - want, axis=1) / size


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(8, 33, 256), (9, 1, 2048), (31, 65, 512), (32, 64, 4096), (33, 500, 2304), (65, 129, 768),
                                   (300, 5200, 256), (70, 7000, 256), (130, 3300, 512), (12, 9000, 256), (3, 60, 512)])
def test_rows_of_every_form(hip, fmt, m, n, k):
    assert errors(hip, fmt, m, n, k, residual=m % 2 == 0).max() <= 1e-6


@pytest.mark.parametrize("fmt", [Q4_0, Q8_0])
@pytest.mark.parametrize("m,n,k", [(8, 17, 32), (40, 70, 288), (9, 40, 1056), (200, 3300, 96)])
def test_rows_that_end_inside_a_chunk(hip, fmt, m, n, k):
    assert errors(hip, fmt, m, n, k).max() <= 1e-6


@pytest.mark.parametrize("fmt", FORMATS)
def test_non_finite_and_tiny_activations(hip, fmt):
    m, n, k = 9, 70, 512
    wq = synth.model_weights(fmt, n, k, 5, 1)
    x = synth.activations(m, k, 6, 1)
    w, t = hip.Tensor.from_numpy(wq), hip.Tensor.from_numpy
    clean = hip.mul_mat_q(fmt, w, n, k, t(x), flags=MATMUL_PRECISE).numpy()
    x[0, 3], x[1, 9], x[2], x[3] = np.inf, np.nan, 0.0, x[3] * np.float32(1e-42)
    got = hip.mul_mat_q(fmt, w, n, k, t(x), flags=MATMUL_PRECISE).numpy()
    assert not np.any(np.isfinite(got[0])) and np.all(np.isnan(got[1])) and np.all(got[2] == 0.0)
    assert np.all(np.abs(got[3]) <= 1e-38)
    assert np.array_equal(got[4:], clean[4:])


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("n,k", [(33, 256), (1, 2048), (70, 2304), (64, 768), (8200, 2048), (500, 4096)])
@pytest.mark.parametrize("m", [2, 3, 4, 5, 6, 7, 8])
def test_few_rows(hip, fmt, m, n, k):
    assert errors(hip, fmt, m, n, k, residual=m % 2 == 0).max() <= 1e-6


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(2, 15, 256), (3, 17, 2304), (5, 4095, 256), (8, 4096, 512), (3, 4097, 512), (4, 4113, 256)])
def test_few_rows_where_the_tile_changes(hip, fmt, m, n, k):
    """Edges of sixteen weight rows, and both sides of the line to 32."""
    assert errors(hip, fmt, m, n, k, residual=m % 2 == 0).max() <= 1e-6


@pytest.mark.parametrize("fmt", [Q4_0, Q8_0])
@pytest.mark.parametrize("m,n,k", [(2, 17, 32), (4, 33, 288), (7, 40, 1056), (3, 70, 2080)])
def test_few_rows_that_end_inside_a_chunk(hip, fmt, m, n, k):
    assert errors(hip, fmt, m, n, k).max() <= 1e-6


@pytest.mark.parametrize("fmt", FORMATS)
def test_few_rows_with_non_finite_and_tiny_activations(hip, fmt):
    m, n, k = 6, 70, 768
    wq = synth.model_weights(fmt, n, k, 5, 1)
    x = synth.activations(m, k, 6, 1)
    w, t = hip.Tensor.from_numpy(wq), hip.Tensor.from_numpy
    clean = hip.mul_mat_q(fmt, w, n, k, t(x), flags=MATMUL_PRECISE).numpy()
    x[0, 3], x[1, 9], x[2], x[3] = np.inf, np.nan, 0.0, x[3] * np.float32(1e-42)
    got = hip.mul_mat_q(fmt, w, n, k, t(x), flags=MATMUL_PRECISE).numpy()
    assert not np.any(np.isfinite(got[0])) and np.all(np.isnan(got[1])) and np.all(got[2] == 0.0)
    assert np.all(np.abs(got[3]) <= 1e-38)
    assert np.array_equal(got[4:], clean[4:])


@pytest.mark.parametrize("fmt,m", [(Q8_0, 3), (Q4_K, 5), (Q6_K, 2)])
def test_few_rows_at_addresses_of_least_alignment(hip, fmt, m):
    """Weights on 2 bytes, activations on 4, each the end of its allocation."""
    n, k = 37, 512
    wq, x = synth.model_weights(fmt, n, k, 5, 3), synth.activations(m, k, 6, 3)
    want = hip.mul_mat_q(fmt, hip.Tensor.from_numpy(wq), n, k, hip.Tensor.from_numpy(x), flags=MATMUL_PRECISE).numpy()
    from litenn_amd import _lib
    w = hip.Tensor.from_numpy(np.concatenate([np.zeros(2, np.uint8), wq.reshape(-1)]))
    xt = hip.Tensor.from_numpy(np.concatenate([np.zeros(1, np.float32), x.reshape(-1)]))
    y = hip.Tensor.from_numpy(np.full((m, n), np.nan, np.float32))
    at = lambda t, o: (t.ptr.value if hasattr(t.ptr, "value") else t.ptr) + o
    _lib.check(_lib.load().litenn_hip_mul_mat_q(0, fmt, at(w, 2), n, k, at(xt, 4), 0, m, y.ptr, None, MATMUL_PRECISE, None))
    assert np.array_equal(y.numpy(), want)


def test_a_workspace_that_holds_the_rows_is_used_and_a_smaller_one_is_enough(hip):
    """The same bits out of the pool's memory and a caller's; with less room the rows go through the streaming kernel."""
    import ctypes as C
    from litenn_amd import _lib
    fmt, m, n, k = Q4_K, 40, 200, 512
    wq = synth.model_weights(fmt, n, k, 5, 2)
    x = synth.activations(m, k, 6, 2)
    w, xt = hip.Tensor.from_numpy(wq), hip.Tensor.from_numpy(x)
    want = hip.mul_mat_q(fmt, w, n, k, xt, flags=MATMUL_PRECISE).numpy()
    for size, same in ((64 * 512 * 5, True), (1024, False)):
        room = hip.Tensor.from_numpy(np.zeros(size, np.uint8))
        y = hip.Tensor.from_numpy(np.full((m, n), np.nan, np.float32))
        _lib.check(_lib.load().litenn_hip_mul_mat_q_ws(0, fmt, w.ptr, n, k, xt.ptr, 0, m, y.ptr, None, MATMUL_PRECISE, room.ptr,
                                                       C.c_size_t(size), None))
        got = y.numpy()
        assert np.array_equal(got, want) == same
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(3, 70, 768), (8, 33, 256), (40, 130, 768), (300, 5200, 512)])
def test_activations_far_below_their_rows_largest_keep_their_bits(hip, fmt, m, n, k):
    """A sub-block of zero weights hides one large activation.  Down to 2^-28 of it an activation is off by 2^-24 of itself at
    most, so that the bound above holds for the others."""
    wq = synth.model_weights(fmt, n, k, 31, m).copy()
    rows = wq.reshape(n, -1)
    if fmt in (Q4_0, Q8_0):
        rows[:, :2] = 0  # the first block's scale
    elif fmt == Q6_K:
        rows[:, 192] = 0  # the first sub-block's scale
    else:
        rows[:, [4, 8]] &= 0xC0  # its scale and its minimum
    w = np_decoders.decode(fmt, wq, k).astype(np.float64)
    assert not w[:, :16].any()
    x = synth.activations(m, k, 32, m)
    x[:, 0] = np.float32(2.0) ** (24 - 7 * np.arange(m) % 25).astype(np.float32)
    got = hip.mul_mat_q(fmt, hip.Tensor.from_numpy(wq), n, k, hip.Tensor.from_numpy(x), flags=MATMUL_PRECISE).numpy()
    rest = x.astype(np.float64)
    rest[:, 0] = 0.0
    size = np.linalg.norm(rest, axis=1) * np.linalg.norm(w) / np.sqrt(k)
    assert (np.linalg.norm(got - rest @ w.T, axis=1) / size).max() <= 1e-6


@pytest.mark.parametrize("fmt", [Q4_K, Q5_K])
@pytest.mark.parametrize("m,n,k", [(6, 70, 768), (40, 130, 512), (300, 5200, 256)])
def test_infinite_activations_give_the_infinities_that_one_row_by_itself_gives(hip, fmt, m, n, k):
    wq = synth.model_weights(fmt, n, k, 5, 4)  # (scales of either sign, so that some sums are infinite and no NaN)
    x = synth.activations(m, k, 6, 4)
    x[0, 3], x[1, 200], x[2, [70, 90]], x[3, [10, 255]] = np.inf, -np.inf, np.inf, [-np.inf, np.inf]
    w, t = hip.Tensor.from_numpy(wq), hip.Tensor.from_numpy
    got = hip.mul_mat_q(fmt, w, n, k, t(x), flags=MATMUL_PRECISE).numpy()
    want = np.concatenate([hip.mul_mat_q(fmt, w, n, k, t(x[i:i + 1]), flags=MATMUL_PRECISE).numpy() for i in range(4)])
    signed = np.isinf(want)  # (where that is no number, the several rows' sums, formed in another order, may be one)
    assert signed.sum() >= 8
    assert np.array_equal(got[:4][signed], want[signed]) and not np.isfinite(got[:4]).any()
    assert np.isfinite(got[4:]).all()


@pytest.mark.parametrize("fmt,m,n,k", [(Q4_K, 9, 40, 256), (Q8_0, 33, 200, 1056), (Q6_K, 64, 70, 512)])
def test_a_workspace_of_the_size_asked_for_is_used(hip, fmt, m, n, k):
    import ctypes as C
    from litenn_amd import _lib
    lib = _lib.load()
    size = lib.litenn_hip_mul_mat_q_precise_workspace_bytes(m, k)
    wq, x = synth.model_weights(fmt, n, k, 5, 2), synth.activations(m, k, 6, 2)
    w, xt = hip.Tensor.from_numpy(wq), hip.Tensor.from_numpy(x)
    want = hip.mul_mat_q(fmt, w, n, k, xt, flags=MATMUL_PRECISE).numpy()
    room = hip.Tensor.from_numpy(np.zeros(size, np.uint8))
    y = hip.Tensor.from_numpy(np.full((m, n), np.nan, np.float32))
    _lib.check(lib.litenn_hip_mul_mat_q_ws(0, fmt, w.ptr, n, k, xt.ptr, 0, m, y.ptr, None, MATMUL_PRECISE, room.ptr, C.c_size_t(size), None))
    assert np.array_equal(y.numpy(), want) and room.numpy().any()


@pytest.mark.parametrize("m,k,some", [(1, 512, False), (8, 512, False), (9, 16384, True), (9, 16640, False), (40, 48, False)])
def test_a_workspace_is_asked_for_where_one_is_used(hip, m, k, some):
    from litenn_amd import _lib
    size = _lib.load().litenn_hip_mul_mat_q_precise_workspace_bytes(m, k)
    assert (size >= 4 * m * k) == some and (size > 0) == some


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(300, 5200, 1280), (300, 2000, 4352), (33, 4100, 4352), (200, 2100, 768), (96, 7000, 512)])
def test_forms_of_two_tiles_over_several_chunks(hip, fmt, m, n, k):
    """Ranges of three chunks and two (four wavefronts on shared activations; two tiles of Q6_K), and sizes beside them."""
    assert errors(hip, fmt, m, n, k, residual=fmt == Q4_0).max() <= 1e-6


# workgroups of 128 x 64 results on both sides of what pays, ranges that are not all alike, a last row and strip of their own
RANGED = [(Q6_K, 300, 2049, 4352), (Q6_K, 257, 2048, 4096), (Q6_K, 33, 10241, 4096), (Q6_K, 70, 16300, 4096), (Q6_K, 100, 4096, 14336),
          (Q4_K, 300, 3300, 7168), (Q5_K, 129, 4097, 7424), (Q4_K, 40, 14336, 4096), (Q5_K, 64, 4000, 14336),
          (Q6_K, 300, 8193, 4096), (Q6_K, 520, 4100, 4352), (Q6_K, 700, 2049, 8448)]


@pytest.mark.parametrize("fmt,m,n,k", RANGED)
def test_ranges_of_k_whose_sums_a_launch_more_adds(hip, fmt, m, n, k):
    """In the call's own memory; a caller's workspace has no room for them."""
    assert errors(hip, fmt, m, n, k, residual=m % 2 == 1).max() <= 1e-6


@pytest.mark.parametrize("fmt,m,n,k", [(Q4_K, 300, 3301, 7168), (Q5_K, 129, 4097, 7424), (Q6_K, 100, 8195, 4096), (Q6_K, 520, 4101, 4352)])
@pytest.mark.parametrize("residual", [False, True])
def test_ranges_of_k_whose_sums_alone_leave_float32(hip, fmt, m, n, k, residual):
    """Sums of ranges beyond Float32's largest value whose sum is not, and sums among its subnormal ones, which are rounded
    once: to half of 2^-149."""
    wq, x = hip.Tensor.from_numpy(synth.model_weights(fmt, n, k, 61)), synth.activations(m, k, 62)
    x[0] = np.sign(x[0]) * np.float32(3e38)
    x[1] *= np.float32(1e-38)
    add = synth.activations(m, n, 63) if residual else np.zeros((m, n), np.float32)
    add[1] *= np.float32(1e-38)
    got = hip.mul_mat_q(fmt, wq, n, k, hip.Tensor.from_numpy(x), residual=hip.Tensor.from_numpy(add) if residual else None, flags=MATMUL_PRECISE).numpy()
    w = np_decoders.decode(fmt, wq.numpy().reshape(n, -1), k).astype(np.float64)
    want = x[:2].astype(np.float64) @ w.T + add[:2]
    size = np.linalg.norm(x[:2].astype(np.float64), axis=1)[:, None] * np.linalg.norm(w, axis=1)
    top = float(np.finfo(np.float32).max)
    fits = np.abs(want[0]) + 1e-6 * size[0] < top
    assert 0.5 < fits.mean() < 0.99
    assert (np.abs(got[0] - want[0]) <= 1e-6 * size[0])[fits].all()
    assert (np.abs(got[1] - want[1]) <= 1e-6 * size[1] + 2.0 ** -150).all()


@pytest.mark.parametrize("fmt,m,n,k,residual", [(Q6_K, 4200, 4099, 4096, True), (Q6_K, 300, 65600, 4096, False)])
def test_ranges_of_k_for_some_rows_at_a_time(hip, fmt, m, n, k, residual):
    """More sums than are left at once: rows in two or three launches, a last one that is not whole; each row as in a call of few."""
    wq, x, add = hip.Tensor.from_numpy(synth.model_weights(fmt, n, k, 71)), synth.activations(m, k, 72), synth.activations(m, n, 73)
    run = lambda rows: hip.mul_mat_q(fmt, wq, n, k, hip.Tensor.from_numpy(x[rows]), residual=hip.Tensor.from_numpy(add[rows]) if residual else None,
                                     flags=MATMUL_PRECISE).numpy()
    got = run(slice(None))
    for first, end in ((0, 70), (m // 2 - 90, m // 2 + 90), (m - 70, m)):  # (beyond 256 workgroups of 128 x 64 results, as all)
        if (n + 127) // 128 * ((end - first + 63) // 64) > 256:
            np.testing.assert_array_equal(got[first:end], run(slice(first, end)))
    w = np_decoders.decode(fmt, wq.numpy().reshape(n, -1), k).astype(np.float64)
    for rows in (slice(0, 8), slice(m // 2 - 8, m // 2 + 8), slice(m - 8, m)):
        size = np.linalg.norm(x[rows].astype(np.float64), axis=1)[:, None] * np.linalg.norm(w) / np.sqrt(n * k) * np.sqrt(k)
        want = x[rows].astype(np.float64) @ w.T + (add[rows] if residual else 0.0)
        assert (np.abs(got[rows] - want) <= 1e-5 * size).all() and np.linalg.norm(got[rows] - want) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("m", [9, 32, 33])
def test_many_weight_rows_meet_one_tile_of_activations(hip, m):
    """More workgroups of 128 x 64 results than CUs: up to 32 rows leave half of each empty and take the form without ranges of K."""
    assert errors(hip, Q6_K, m, 32801, 4096).max() <= 1e-6


@pytest.mark.parametrize("fmt,m,n,k", RANGED[4:8])
def test_infinite_activations_in_ranges_of_k(hip, fmt, m, n, k):
    wq, x = hip.Tensor.from_numpy(synth.model_weights(fmt, n, k, 61)), synth.activations(m, k, 62)
    run = lambda rows: hip.mul_mat_q(fmt, wq, n, k, hip.Tensor.from_numpy(rows), flags=MATMUL_PRECISE).numpy()
    clean = run(x)
    x[3, 5], x[4, k - 1], x[m - 1, k // 2] = np.inf, -np.inf, np.nan
    got = run(x)
    assert np.isnan(got[m - 1]).all() and not np.isfinite(got[3:5]).any()
    for row in (3, 4) if fmt == Q4_K else ():  # (one row of the others may take an infinity off an infinite sum)
        np.testing.assert_array_equal(got[row], run(x[row:row + 1])[0])
    rest = [i for i in range(m) if i not in (3, 4, m - 1)]
    np.testing.assert_array_equal(got[rest], clean[rest])


@pytest.mark.parametrize("fmt", [Q4_K, Q5_K])
@pytest.mark.parametrize("n,k", [(5185, 256), (5200, 768), (5200, 4352)])
def test_one_range_of_k_adds_as_two(hip, fmt, n, k):
    """More than 256 workgroups go over K in one range, fewer in two: a row's sums are the same bits."""
    wq, x = hip.Tensor.from_numpy(synth.model_weights(fmt, n, k, 51)), synth.activations(450, k, 52)
    run = lambda rows: hip.mul_mat_q(fmt, wq, n, k, hip.Tensor.from_numpy(rows), flags=MATMUL_PRECISE).numpy()
    got = run(x)
    np.testing.assert_array_equal(got[:300].view(np.uint32), run(x[:300]).view(np.uint32))
    w = np_decoders.decode(fmt, wq.numpy().reshape(n, -1), k).astype(np.float64)
    size = np.linalg.norm(x.astype(np.float64), axis=1) * np.linalg.norm(w) / np.sqrt(k)
    assert (np.linalg.norm(got - x.astype(np.float64) @ w.T, axis=1) / size).max() <= 1e-6


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,k", [(3, 256), (3, 4096), (45, 4096)])
def test_several_rows_are_no_further_off_than_rows_one_by_one(hip, fmt, m, k):
    """Error against 64 bits, mean of six inputs."""
    n, many, one = 300, [], []
    T = hip.Tensor.from_numpy
    for seed in range(6):
        wq, x = synth.model_weights(fmt, n, k, 40, seed), synth.activations(m, k, 41, seed)
        w, want = T(wq), x.astype(np.float64) @ np_decoders.decode(fmt, wq, k).astype(np.float64).T
        off = lambda got: np.linalg.norm(got - want) / np.linalg.norm(want)
        many.append(off(hip.mul_mat_q(fmt, w, n, k, T(x), flags=MATMUL_PRECISE).numpy()))
        one.append(off(np.concatenate([hip.mul_mat_q(fmt, w, n, k, T(x[i:i + 1]), flags=MATMUL_PRECISE).numpy() for i in range(m)])))
    assert np.mean(many) <= np.mean(one)
