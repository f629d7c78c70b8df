"""GPU parity of the many-row product with superblock weights (Q4_K, Q5_K, Q6_K) and blocks of 32 (Q4_0, Q4_1, Q5_0, Q5_1, Q8_0):
every tile it has, at its edges, against the float64 product of the dequantised weights.

Bound: an f32 row keeps 22 bits (2^-23 of each element) and K products are added in f32, in at most 4 K / 256 + 8 parts whose
sums are rounded: |error| <= (2^-22 + (K / 64 + 8) 2^-24) sum |x w|, and the change of the accumulators' unit rounds them once
more per superblock.  Three times that is allowed."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.util import gen_weight

pytestmark = pytest.mark.gpu


def _check(ctx, qtype, n, k, packed, x, bias=None, bf16=False):
    deq = o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64)
    qt = q.QuantizedTensor([n, k], qtype, packed)
    if bf16:
        xb = q.f32_to_bf16_bits(x)
        got, x = q.quantized_matmul_bf16(xb, qt, ctx), q.bf16_bits_to_f32(xb)
    else:
        got = q.quantized_matmul(x, qt, bias, ctx)
    x = x.astype(np.float64)
    want = x @ deq.T + (0 if bias is None else bias.astype(np.float64))
    # types with an offset are added as two parts, each as large as the codes' range
    span = 3.0 if qtype in (o.Q4_K, o.Q5_K, o.Q4_1, o.Q5_1) else 1.0
    bound = 3 * (2.0 ** -22 + (k / 64 + 8) * 2.0 ** -24) * span * (np.abs(x) @ np.abs(deq).T) + 2.0 ** -22 * np.abs(want) + 1e-30
    off = np.abs(got - want) / bound
    assert np.isfinite(got).all() and off.max() <= 1, f"{o.TYPE_NAMES[qtype]} {x.shape[0]} x {n} x {k}: {off.max():.2f} of the bound"


BLOCKS = [o.Q4_0, o.Q4_1, o.Q5_0, o.Q5_1, o.Q8_0]


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K, *BLOCKS])
@pytest.mark.parametrize("rows,n,k", [(9, 1, 256), (10, 1, 256), (16, 128, 512), (17, 129, 768), (32, 127, 2304), (33, 260, 256), (39, 132, 1280),
                                      (48, 64, 4352), (64, 128, 1024), (65, 257, 512), (128, 256, 256), (130, 4, 768), (10, 2048, 4096), (40, 1030, 2560)])
def test_tiles_and_remainders(ctx, qtype, rows, n, k):
    """Row counts on both sides of the tiles of 16, 32, 39, 64 and 128 f32 rows, columns around 128 and 256, one superblock, odd counts
    of them for the two halves of a workgroup, and K in pieces."""
    rng = np.random.default_rng(rows * 7 + n + k + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    x = rng.standard_normal((rows, k)).astype(np.float32) * (10.0 ** rng.integers(-3, 4, size=(rows, 1))).astype(np.float32)
    _check(ctx, qtype, n, k, packed, x, bias=rng.standard_normal(n).astype(np.float32))
    _check(ctx, qtype, n, k, packed, x, bf16=True)


@pytest.mark.parametrize("qtype,size,at", [(o.Q4_K, 144, 0), (o.Q5_K, 176, 0), (o.Q6_K, 210, 208)])
@pytest.mark.parametrize("rows", [12, 24, 56, 160])
def test_superblocks_of_every_scale(ctx, qtype, size, at, rows):
    """Superblocks without a scale, without a minimum, with neither, with a minimum far above the scale and of either sign: the
    accumulators' unit changes by up to 2^40 between neighbours."""
    rng = np.random.default_rng(rows + qtype)
    n, k = 140, 1536
    b = o.quantize(qtype, gen_weight(rng, n, k)).reshape(-1, size).copy()
    d = np.array([0, 6e-8, 1e-6, 1e-3, 0.5, 300, -1e-3], np.float16)
    m = np.array([0, 0, 6e-8, 1e-4, 0.1, 60, -0.05], np.float16)
    b[:, at:at + 2] = rng.choice(d, len(b)).view(np.uint8).reshape(-1, 2)
    if qtype != o.Q6_K:
        b[:, 2:4] = rng.choice(m, len(b)).view(np.uint8).reshape(-1, 2)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[1] = np.abs(x[1])
    _check(ctx, qtype, n, k, b.reshape(-1), x)


@pytest.mark.parametrize("qtype,size", [(o.Q4_K, 144), (o.Q5_K, 176)])
@pytest.mark.parametrize("rows", [12, 24, 39, 56, 100, 160])
@pytest.mark.parametrize("k", [256, 768])
def test_every_pair_of_scale_and_minimum(ctx, qtype, size, rows, k):
    """Scales and minima of every power of two that f16 has, 2^-24 to 2^15, in all pairs, and of either sign: a column of its own for
    a pair, and three pairs to a column."""
    rng = np.random.default_rng(rows + k + qtype)
    e = np.arange(-24, 16)
    d, m = (v.ravel() for v in np.meshgrid(e, e))
    n, per = len(d), k // 256
    b = o.quantize(qtype, gen_weight(rng, n, k)).reshape(n, per, size).copy()
    for s in range(per):
        order = rng.permutation(n) if s else np.arange(n)
        for at, v in ((0, d[order]), (2, m[order])):
            f = np.minimum(2.0 ** v * (1 + rng.random(n)), 65504.0) * rng.choice([1.0, 1.0, -1.0], n)
            b[:, s, at:at + 2] = f.astype(np.float16).view(np.uint8).reshape(n, 2)
    _check(ctx, qtype, n, k, b.reshape(-1), rng.standard_normal((rows, k)).astype(np.float32))


@pytest.mark.parametrize("qtype", BLOCKS)
@pytest.mark.parametrize("rows,n", [(129, 257), (513, 640), (130, 16384), (130, 16385)])
def test_blocks_in_many_tiles(ctx, qtype, rows, n):
    """More than one tile of rows, K in pieces or whole; as many tiles as compute units with bf16 rows (2 x 128) and
    one column more, which the large tiles take (several superblocks of those: test_gpu_gemm_rows_large.py)."""
    k = 256 if n > 10000 else 1536
    rng = np.random.default_rng(rows + n + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    x = rng.standard_normal((rows, k)).astype(np.float32)
    _check(ctx, qtype, n, k, packed, x, bf16=True)
    if n < 10000:
        _check(ctx, qtype, n, k, packed, x)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K, *BLOCKS])
@pytest.mark.parametrize("rows,n,k", [(10, 100, 8192), (16, 4096, 4352), (16, 4100, 4096), (17, 100, 8192), (24, 260, 14336), (33, 132, 8192)])
def test_few_rows_on_both_sides_of_the_gemv(ctx, qtype, rows, n, k):
    """Ten to sixteen rows that the small-batch GEMV keeps or hands over by type, weight rows and K; K in sixteen parts."""
    rng = np.random.default_rng(rows + n + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    _check(ctx, qtype, n, k, packed, rng.standard_normal((rows, k)).astype(np.float32), bias=rng.standard_normal(n).astype(np.float32))


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K])
@pytest.mark.parametrize("rows,n,k,bf16", [(129, 8192, 256, True), (129, 8193, 256, True), (257, 8129, 768, True), (300, 5377, 1280, False), (2047, 1000, 8192, True)])
def test_superblocks_in_large_tiles(ctx, qtype, rows, n, k, bf16):
    """As many tiles of 128 x 128 as half the compute units, and more, which 256 x 256 outputs take; and few outputs over a K that is
    long enough for eight parts."""
    rng = np.random.default_rng(rows + n + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    _check(ctx, qtype, n, k, packed, rng.standard_normal((rows, k)).astype(np.float32), bf16=bf16)


@pytest.mark.parametrize("qtype", BLOCKS)
@pytest.mark.parametrize("rows", [12, 24, 56])
def test_blocks_of_every_scale(ctx, qtype, rows):
    """Blocks without a scale, without a minimum, with neither, from f16's smallest numbers to its largest, of either sign."""
    rng = np.random.default_rng(rows + qtype)
    n, k = 140, 1536
    size = {o.Q4_0: 18, o.Q4_1: 20, o.Q5_0: 22, o.Q5_1: 24, o.Q8_0: 34}[qtype]
    b = o.quantize(qtype, gen_weight(rng, n, k)).reshape(-1, size).copy()
    d = np.array([0, 6e-8, 1e-6, 1e-3, 0.5, 300, -1e-3, 65504 if qtype != o.Q5_1 else 2000], np.float16)
    b[:, :2] = rng.choice(d, len(b)).view(np.uint8).reshape(-1, 2)
    if qtype in (o.Q4_1, o.Q5_1):
        m = np.array([0, 0, 6e-8, 1e-4, -0.1, 60, -65504], np.float16)
        b[:, 2:4] = rng.choice(m, len(b)).view(np.uint8).reshape(-1, 2)
    b[:k // 32, :2] = 0  # a row of nothing but minima
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[1] = np.abs(x[1])
    _check(ctx, qtype, n, k, b.reshape(-1), x)


def test_zero_rows_and_rows_of_extreme_magnitude(ctx):
    rng = np.random.default_rng(1)
    n, k = 130, 512
    packed = o.quantize(o.Q4_K, gen_weight(rng, n, k))
    x = rng.standard_normal((20, k)).astype(np.float32)
    x[0], x[3], x[4] = 0, x[3] * 1e30, x[4] * 1e-30
    _check(ctx, o.Q4_K, n, k, packed, x)
    x[5, 7], x[6, 9] = np.inf, np.nan
    got = q.quantized_matmul(x, q.QuantizedTensor([n, k], o.Q4_K, packed), None, ctx)
    assert not np.isfinite(got[5]).any() and np.isnan(got[6]).all()  # and nothing of them in other rows
    keep = [r for r in range(20) if r not in (5, 6)]
    assert np.isfinite(got[keep]).all()
