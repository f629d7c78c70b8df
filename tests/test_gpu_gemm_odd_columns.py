"""Products of a number of columns that is no multiple of four, K in parts: every tile of the many-row kernels, partial sums and their reduction
at the last columns, and the same calls where there is no room for the parts.

Bound: 3e-7 of the results' root mean square for the f32 sums (1e-7 is measured, see test_gpu_gemm_rows_uneven), f32 rows as pairs of f16 (22 bits) and
16-bit weights through two planes included: 2^-22 sqrt(2)."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.util import gen_weight

pytestmark = pytest.mark.gpu


def _check(ctx, qtype, rows, n, k, bf16):
    rng = np.random.default_rng(rows + n + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    w = o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64)
    qt = q.QuantizedTensor([n, k], qtype, packed)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    if bf16:
        bits = q.f32_to_bf16_bits(x)
        got, want = q.quantized_matmul_bf16(bits, qt, ctx), q.bf16_bits_to_f32(bits).astype(np.float64) @ w.T
    else:
        got, want = q.quantized_matmul(x, qt, bias, ctx), x.astype(np.float64) @ w.T + bias
    rms = lambda v: np.sqrt(np.mean(np.square(v)))
    assert rms(got - want) <= (3e-7 + 2.0 ** -22 * 2 ** 0.5) * rms(want)
    edge = np.s_[:, n // 4 * 4 - 4:]  # the last whole group of columns and what is left
    assert rms((got - want)[edge]) <= 2 * (3e-7 + 2.0 ** -22 * 2 ** 0.5) * rms(want)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q6_K, o.Q5_1, o.Q8_0, o.F16])
@pytest.mark.parametrize("n", [129, 258, 515])
@pytest.mark.parametrize("rows,bf16", [(10, False), (32, False), (39, False), (47, False), (150, False), (24, True), (64, True), (128, True), (700, True)])
def test_odd_columns(ctx, qtype, n, rows, bf16):
    _check(ctx, qtype, rows, n, 2048, bf16)


@pytest.mark.parametrize("qtype,k", [(o.Q5_K, 14336), (o.Q4_0, 8192), (o.Q4_1, 1024 + 64)])
def test_odd_columns_of_long_and_ragged_rows(ctx, qtype, k):
    _check(ctx, qtype, 100, 1027, k, True)
    _check(ctx, qtype, 50, 1027, k, False)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.F16])
def test_without_room_for_the_parts_of_k(monkeypatch, qtype):
    ctx = q.Context(0)
    room = 2 * 128 * 2048 * 2  # the rows' operands (twice, their sums and scales with them), not eight parts of 128 x 515
    monkeypatch.setenv("AXQ_GEMM_SCRATCH_MAX", str(room))
    _check(ctx, qtype, 100, 515, 2048, True)
    monkeypatch.delenv("AXQ_GEMM_SCRATCH_MAX")
    _check(ctx, qtype, 100, 515, 2048, True)
