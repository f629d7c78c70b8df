"""GPU parity of the many-row product on rows with elements far above the others, as activations have: the large ones meet weights of
zero, so that what the small ones lose shows in the result.

Bound: the root mean square of the error over all results stays within that of sum_k delta_k w_k, delta_k the largest error of element k
in the kernels' operands, plus 3e-7 of the results' for the f32 sums (1e-7 is measured).  With the row's largest element in
[2^t, 2^(t + 1)):
  rows of f16 pairs   delta = 2^-22 |x| + 2^(t - 39): f16's smallest number is 2^-38 of the largest power of two
  bf16 rows           delta = 2^(t - 39)
  rows of limbs       delta = min(2^-22 |x|, 2^(g - 31)) + 2^(t - 48), 2^g the power of two of the largest of the element's 32
Where weights have an offset, the offset of 32 of them (at most the middle of their range and half a step) meets a sum of x that is
off by as much as 2^(t - 33), or 2^(t - 42) with limbs."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.util import gen_weight

pytestmark = pytest.mark.gpu

LIMBS = 40  # f32 rows below it are limbs
TYPES = [o.Q4_K, o.Q5_K, o.Q6_K, o.Q4_0, o.Q4_1, o.Q5_0, o.Q5_1, o.Q8_0]
SYMMETRIC = [o.Q4_0, o.Q5_0, o.Q8_0, o.Q6_K]  # a single weight can be zero exactly


def _power(v):
    return np.floor(np.log2(np.abs(v)))


def _check(ctx, qtype, x, n, zero, bf16=False):
    """`zero`: the places along K whose weights are zero and whose elements of x are the large ones."""
    rng = np.random.default_rng(x.shape[0] + n + qtype)
    rows, k = x.shape
    w = gen_weight(rng, n, k)
    w[:, zero] = 0
    packed = o.quantize(qtype, w)
    w = o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64)
    assert not w[:, zero].any()
    qt = q.QuantizedTensor([n, k], qtype, packed)
    if bf16:
        bits = q.f32_to_bf16_bits(x)
        got, x = q.quantized_matmul_bf16(bits, qt, ctx), q.bf16_bits_to_f32(bits)
    else:
        got = q.quantized_matmul(x, qt, None, ctx)
    x = x.astype(np.float64)
    want = x @ w.T
    t = _power(np.abs(x).max(1, keepdims=True))
    if bf16:
        delta = np.broadcast_to(2.0 ** (t - 39), x.shape)
    elif rows < LIMBS:
        g = np.repeat(_power(np.abs(x).reshape(rows, k // 32, 32).max(2)), 32, axis=1)
        delta = np.minimum(2.0 ** -22 * np.abs(x), 2.0 ** (g - 31)) + 2.0 ** (t - 48)
    else:
        delta = 2.0 ** -22 * np.abs(x) + 2.0 ** (t - 39)
    square = delta ** 2 @ (w ** 2).T
    if qtype not in SYMMETRIC:
        b = w.reshape(n, k // 32, 32)
        lo, hi = b.min(2), b.max(2)
        offset = np.abs(lo + hi) / 2 + (hi - lo) / 30
        square += 4.0 ** (t - (33 if bf16 or rows >= LIMBS else 42)) * (offset ** 2).sum(1)
    rms = lambda v: np.sqrt(np.mean(np.square(v)))
    off, bound = rms(got - want), np.sqrt(np.mean(square)) + 3e-7 * rms(want)
    assert off <= bound, f"{o.TYPE_NAMES[qtype]} {rows} x {n} x {k}: {off / rms(want):.2e}, bound {bound / rms(want):.2e}"


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("rows", [10, 16, 17, 32, 33, 39, 40, 64, 65, 160])
@pytest.mark.parametrize("top", [14, 23])
def test_a_large_element_in_a_block_of_its_own(ctx, qtype, rows, top):
    rng = np.random.default_rng(rows + top)
    x = rng.standard_normal((rows, 1024)).astype(np.float32)
    x[np.arange(rows), 256 + rng.integers(0, 32, size=rows)] = 1.5 * 2.0 ** top
    _check(ctx, qtype, x, 384, np.arange(256, 288))


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("rows", [10, 64, 130, 300])
@pytest.mark.parametrize("top", [20, 29])
def test_bf16_rows_with_a_large_element(ctx, qtype, rows, top):
    rng = np.random.default_rng(rows + top)
    x = rng.standard_normal((rows, 1024)).astype(np.float32)
    x[np.arange(rows), 256 + rng.integers(0, 32, size=rows)] = 1.5 * 2.0 ** top
    _check(ctx, qtype, x, 384, np.arange(256, 288), bf16=True)


@pytest.mark.parametrize("qtype", SYMMETRIC)
@pytest.mark.parametrize("rows", [10, 16, 17, 32, 33, 39, 40, 64])
@pytest.mark.parametrize("top", [9, 14])
def test_a_large_element_in_every_block(ctx, qtype, rows, top):
    """Below 40 rows the second and the third limb carry the small elements."""
    rng = np.random.default_rng(rows + top)
    x = rng.standard_normal((rows, 1024)).astype(np.float32)
    x[:, 7::32] = 1.5 * 2.0 ** top
    _check(ctx, qtype, x, 384, np.arange(7, 1024, 32))


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("rows", [10, 16, 17, 32, 33, 39])
def test_blocks_of_uneven_magnitude(ctx, qtype, rows):
    """Blocks of 32 whose magnitudes lie up to 2^20 apart; the larger half meets weights of zero."""
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, 1024)).astype(np.float32) * np.repeat(2.0 ** -rng.permuted(np.tile(np.arange(8, 17), 4)[:32]), 32).astype(np.float32)
    x[:, 512:] *= np.float32(2.0 ** 12)
    _check(ctx, qtype, x, 384, np.arange(512, 1024))


@pytest.mark.parametrize("qtype,limbs,pairs", [(o.Q4_0, 5.0, 8.3), (o.Q5_1, 6.3, 8.5), (o.Q4_K, 7.3, 11.0), (o.Q6_K, 5.2, 12.1), (o.Q8_0, 7.1, 8.6)])
@pytest.mark.parametrize("rows", [10, 24, 39, 48, 100])
def test_error_of_even_rows(ctx, qtype, limbs, pairs, rows):
    """Root mean square error over that of the results, in 1e-8, against what was measured, a quarter more allowed (the kernels that had
    these calls before it: 8.6 to 10.5 below 40 rows, 10.6 to 21.6 from there on)."""
    rng = np.random.default_rng(rows + qtype)
    n, k = 1024, 4096
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    x = rng.standard_normal((rows, k)).astype(np.float32)
    want = x.astype(np.float64) @ o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64).T
    got = q.quantized_matmul(x, q.QuantizedTensor([n, k], qtype, packed), None, ctx)
    off = np.sqrt(np.mean((got - want) ** 2) / np.mean(want ** 2)) * 1e8
    assert off <= 1.25 * (limbs if rows < LIMBS else pairs), f"{off:.1f}"
