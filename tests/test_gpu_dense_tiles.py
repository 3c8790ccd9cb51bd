"""Products over bfloat16 weights at the edges of the rules that pick a tile and of the K walk (a single step of 64, odd
numbers of steps, ragged K; with Float32 operands two groups of wavefronts may share it), in both operand types.

Bounds: bfloat16 operands are exact, Float32 ones are taken apart exactly, so what is left are Float32 sums of k
products, about sqrt(log2 k) 2^-24 of |x| |W| / sqrt(k); 1e-6 is four times what is seen."""
import numpy as np
import pytest

from litenn_amd.model import from_bfloat16
from test_gpu_layer_ops import NAN16, NAN32, bf16_tensor, padded_bits, pitch

pytestmark = pytest.mark.gpu

# the forms of csrc/fetch_model.hpp that they take (tests/test_cpp_host.py holds SHAPES to all of Float32's, SAME_BITS to
# most of bfloat16's)
SHAPES = [(49200, 64, 65), (12300, 200, 129), (12290, 100, 250),                   # Float32 64 x 256
          (11264, 200, 500), (11200, 205, 760), (11200, 64, 500),                  # 64 x 128 as one chain
          (6200, 320, 250),                                                        # 64 x 128 on two groups
          (3137, 192, 193),                                                        # 64 x 64 on two groups
          (6210, 3100, 130), (3100, 64, 200), (40, 64, 33), (700, 1088, 40), (1030, 4096, 7)]  # 32 x 64 on two groups
SAME_BITS, SAME_BITS_K = (5632, 1430, 20, 43, 100, 150, 250, 270, 330, 500, 710, 970, 1031), (130, 300, 500)


@pytest.mark.parametrize("n,k,m", SHAPES)
@pytest.mark.parametrize("f32", [True, False])
def test_tiles(hip, f32, n, k, m):
    rng = np.random.default_rng([n, k, m])
    w = padded_bits(rng.normal(0, 1, (n, k)).astype(np.float32))
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    wf = from_bfloat16(w)[:, :k].astype(np.float64)
    if f32:
        padded = np.full((m, pitch(k)), NAN32, np.float32)
        padded[:, :k] = x
        xt = hip.Tensor.from_numpy(padded)
    else:
        bits = padded_bits(x, NAN16)
        x = from_bfloat16(bits)[:, :k]
        xt = bf16_tensor(hip, bits)
    got = hip.linear_bf16(bf16_tensor(hip, w), n, k, xt, m).numpy()
    size = np.linalg.norm(x.astype(np.float64), axis=1) * np.linalg.norm(wf) / np.sqrt(k)
    assert (np.linalg.norm(got - x.astype(np.float64) @ wf.T, axis=1) / size).max() <= 1e-6


@pytest.mark.parametrize("k", SAME_BITS_K)
def test_bfloat16_rows_are_the_same_bits_in_every_form(hip, k):
    """A row's sums run over K in one order, however many rows go with it: from 192 x 128 at 1430 rows to 32 x 32 at 20."""
    n, rows, *fewer = SAME_BITS
    rng = np.random.default_rng(k)
    w, x = (padded_bits(rng.normal(0, 1, (r, k)).astype(np.float32)) for r in (n, rows))
    wt = bf16_tensor(hip, w)
    want = hip.linear_bf16(wt, n, k, bf16_tensor(hip, x), rows).numpy()
    exact = from_bfloat16(x)[:9].astype(np.float64) @ from_bfloat16(w).astype(np.float64).T
    assert np.linalg.norm(want[:9] - exact) <= 1e-6 * np.linalg.norm(exact)
    for m in fewer:
        assert np.array_equal(hip.linear_bf16(wt, n, k, bf16_tensor(hip, x[:m]), m).numpy(), want[:m]), m


def test_float32_extremes_stay_in_their_rows(hip):
    """The largest and smallest magnitudes, infinities and NaN (also one whose payload lies in the low bits only)."""
    n, k, m = 96, 128, 40
    rng = np.random.default_rng(1)
    w = padded_bits(rng.normal(0, 1e-3, (n, k)).astype(np.float32))
    wf = from_bfloat16(w).astype(np.float64)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    x[0] *= np.float32(1e38)
    x[1] *= np.float32(1e-30)
    x[2, 5] = np.finfo(np.float32).max
    x[3, 7] = np.inf
    x[4, 9] = np.array([0x7F800001], np.uint32).view(np.float32)[0]
    wt = bf16_tensor(hip, w)
    got = hip.linear_bf16(wt, n, k, hip.Tensor.from_numpy(x), m).numpy()
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ wf.T
    assert np.all(np.isinf(got[3]) & (np.sign(got[3]) == np.sign(wf[:, 7]))) and np.all(np.isnan(got[4]))
    for i in (0, 1, 2, *range(5, m)):
        assert np.linalg.norm(got[i] - want[i]) <= 1e-6 * np.linalg.norm(x[i].astype(np.float64)) * np.linalg.norm(wf) / np.sqrt(k)
