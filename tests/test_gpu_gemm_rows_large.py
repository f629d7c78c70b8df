"""GPU parity of the many-row product in its large tiles (256 x 256 and 256 x 128 outputs, and 128 x 128 whose halves have K of their own), which
calls reach with more tiles than small ones have: K that the rings of x and codes go round in, scales and minima of every size, infinities."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.decode_common import load_gpu, random_weights, tiny_config
from tests.test_gpu_gemm_rows import BLOCKS, _check
from tests.util import gen_weight

pytestmark = pytest.mark.gpu

SIZE = {o.Q4_K: 144, o.Q5_K: 176, o.Q6_K: 210, o.Q4_0: 18, o.Q4_1: 20, o.Q5_0: 22, o.Q5_1: 24, o.Q8_0: 34}
# rows, columns, K and whether the rows are bf16, of a call for every kernel; APART: K in parts, which are too short for that kernel, and whole, by more than 128 tiles
WIDE = [(600, 1600, 768, False), (1160, 1600, 1024, True)]
APART = [(50, 1601, 2048, False), (100, 1601, 2304, True), (50, 16387, 2048, False), (100, 16387, 2304, True)]
BLOCK32 = [(130, 16500, 768, True), (257, 11009, 1024, True), (130, 16499, 2304, False), (65, 16500, 1024, False)]


def _packed(qtype, rng, n, k, distinct=1009):
    """Rows of weights, some of them again and again."""
    rows = o.quantize(qtype, gen_weight(rng, min(n, distinct), k)).reshape(min(n, distinct), -1)
    return rows[np.arange(n) % len(rows)].copy()


@pytest.mark.parametrize("qtype", BLOCKS)
@pytest.mark.parametrize("rows,n,k,bf16", BLOCK32)
def test_blocks_of_several_superblocks(ctx, qtype, rows, n, k, bf16):
    rng = np.random.default_rng(rows + n + k + qtype)
    x = rng.standard_normal((rows, k)).astype(np.float32) * (10.0 ** rng.integers(-3, 4, size=(rows, 1))).astype(np.float32)
    _check(ctx, qtype, n, k, _packed(qtype, rng, n, k).reshape(-1), x, bias=None if bf16 else rng.standard_normal(n).astype(np.float32), bf16=bf16)


@pytest.mark.parametrize("qtype", BLOCKS)
@pytest.mark.parametrize("rows,n,k,bf16", BLOCK32[:1] + BLOCK32[-1:])
def test_blocks_of_every_scale(ctx, qtype, rows, n, k, bf16):
    rng = np.random.default_rng(rows + qtype)
    b = _packed(qtype, rng, n, k)
    f = b.reshape(-1, SIZE[qtype])
    d = np.array([0, 6e-8, 1e-6, 1e-3, 0.5, 300, -1e-3, 65504 if qtype != o.Q5_1 else 2000], np.float16)
    f[:, :2] = rng.choice(d, len(f)).view(np.uint8).reshape(-1, 2)
    if qtype in (o.Q4_1, o.Q5_1):
        m = np.array([0, 0, 6e-8, 1e-4, -0.1, 60, -65504], np.float16)
        f[:, 2:4] = rng.choice(m, len(f)).view(np.uint8).reshape(-1, 2)
    f[:k // 32, :2] = 0  # a row of nothing but minima
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[1] = np.abs(x[1])
    _check(ctx, qtype, n, k, b.reshape(-1), x, bf16=bf16)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K])
@pytest.mark.parametrize("rows,n,k,bf16", WIDE + APART)
def test_superblocks_of_every_scale(ctx, qtype, rows, n, k, bf16):
    """Also no scale, no minimum, neither, a minimum far above the scale."""
    rng = np.random.default_rng(rows + qtype)
    b = _packed(qtype, rng, n, k, n)
    f, at = b.reshape(-1, SIZE[qtype]), 208 if qtype == o.Q6_K else 0
    f[:, at:at + 2] = rng.choice(np.array([0, 6e-8, 1e-6, 1e-3, 0.5, 300, -1e-3], np.float16), len(f)).view(np.uint8).reshape(-1, 2)
    if qtype != o.Q6_K:
        f[:, 2:4] = rng.choice(np.array([0, 0, 6e-8, 1e-4, 0.1, 60, -0.05], np.float16), len(f)).view(np.uint8).reshape(-1, 2)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[1] = np.abs(x[1])
    _check(ctx, qtype, n, k, b.reshape(-1), x, bf16=bf16)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K])
@pytest.mark.parametrize("rows,n,k,bf16", WIDE + APART)
def test_every_pair_of_scale_and_minimum(ctx, qtype, rows, n, k, bf16):
    """Every power of two that f16 has, 2^-24 to 2^15, in all 1600 pairs, and of either sign."""
    rng = np.random.default_rng(rows + k + qtype)
    d, m = (v.ravel() for v in np.meshgrid(np.arange(-24, 16), np.arange(-24, 16)))
    b = _packed(qtype, rng, n, k, n)
    f = b.reshape(n, k // 256, SIZE[qtype])
    for s in range(k // 256):
        order = np.arange(n) % 1600 if s == 0 else rng.permutation(n) % 1600
        for at, v in ((0, d[order]), (2, m[order])):
            e = np.minimum(2.0 ** v * (1 + rng.random(n)), 65504.0) * rng.choice([1.0, 1.0, -1.0], n)
            f[:, s, at:at + 2] = e.astype(np.float16).view(np.uint8).reshape(n, 2)
    _check(ctx, qtype, n, k, b.reshape(-1), rng.standard_normal((rows, k)).astype(np.float32), bf16=bf16)


@pytest.mark.parametrize("qtype,shape", [(t, s) for t in (o.Q4_K, o.Q5_K, o.Q6_K) for s in WIDE + APART] + [(t, s) for t in BLOCKS for s in BLOCK32[:1] + BLOCK32[-1:]])
def test_infinities_stay_in_their_row_and_column(ctx, qtype, shape):
    rows, n, k, bf16 = shape
    rng = np.random.default_rng(n + qtype)
    b = _packed(qtype, rng, n, k)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[5, 7], x[6, 9] = np.inf, np.nan
    row, at = b.reshape(n, -1, SIZE[qtype]), 208 if qtype == o.Q6_K else 0
    row[40, 1, at:at + 2] = np.array([np.inf], np.float16).view(np.uint8)
    row[n - 1, 0, at:at + 2] = np.array([np.nan], np.float16).view(np.uint8)
    qt = q.QuantizedTensor([n, k], qtype, b.reshape(-1))
    got = q.quantized_matmul_bf16(q.f32_to_bf16_bits(x), qt, ctx) if bf16 else q.quantized_matmul(x, qt, None, ctx)
    assert not np.isfinite(got[5]).any() and np.isnan(got[6]).all() and not np.isfinite(got[:, 40]).any() and np.isnan(got[:, n - 1]).all()
    assert np.isfinite(np.delete(np.delete(got, [5, 6], 0), [40, n - 1], 1)).all()


@pytest.mark.parametrize("qtype", [o.Q4_1, o.Q8_0, o.Q4_K])
def test_residuals_of_a_prompt(ctx, monkeypatch, qtype):
    """The second layer's keys and values of all rows, which come through products with residuals: a prompt in one portion, whose products take
    large tiles, against portions of 64."""
    c = tiny_config(hidden_size=1536, intermediate_size=512, num_heads=12, num_kv_heads=3, head_dim=128, max_seq_len=2100)
    w = random_weights(c, 3, qtype, std=0.02)
    tokens = np.random.default_rng(1).integers(0, c["vocab_size"], size=2048)
    caches = []
    for chunk in ("64", "2048"):
        monkeypatch.setenv("AXQ_PROMPT_CHUNK", chunk)
        gpu = load_gpu(ctx, c, w)
        gpu.forward_tokens(tokens, want_logits=False)
        caches.append([gpu.kv(1, which)[:, :2048].view(np.float16).astype(np.float64) for which in (0, 1)])
        gpu.close()
    for a, b in zip(*caches):
        assert np.abs(a - b).max() <= 2e-3 * np.abs(a).max()  # two roundings to f16 of values that are off by f32's


@pytest.mark.parametrize("qtype,limit", [(o.Q4_0, 21.0), (o.Q4_1, 22.4), (o.Q5_0, 21.0), (o.Q5_1, 22.4), (o.Q8_0, 21.1), (o.Q4_K, 31.4), (o.Q5_K, 32.1), (o.Q6_K, 40.8)])
def test_error_of_even_rows(ctx, qtype, limit):
    """Root mean square error over that of the results, in 1e-8, against what was measured, a quarter more allowed: f32 rows, K = 4096."""
    rng = np.random.default_rng(qtype)
    rows, n, k = 130, 11100, 4096
    packed = _packed(qtype, rng, n, k)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    want = x.astype(np.float64) @ o.dequantize(qtype, packed[:1009].reshape(-1), 1009 * k).reshape(1009, k).astype(np.float64).T
    got = q.quantized_matmul(x, q.QuantizedTensor([n, k], qtype, packed.reshape(-1)), None, ctx)
    off = np.sqrt(np.mean((got - want[:, np.arange(n) % 1009]) ** 2) / np.mean(want ** 2)) * 1e8
    assert off <= 1.25 * limit, f"{off:.1f}"
