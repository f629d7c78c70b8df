"""Weights of blocks of 32 whose rows are no whole superblocks of 256: scales of zero lie behind a row's last one on the device.  Upload and download give the same
bytes, and products of every number of rows agree with 64 bits.

Bound: 3e-7 of the results' root mean square for the f32 sums, f32 rows from 40 on as pairs of f16: 2^-22 sqrt(2) (see test_gpu_gemm_rows_uneven)."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.util import gen_weight

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TYPES = [o.Q4_0, o.Q4_1, o.Q5_0, o.Q5_1, o.Q8_0]


def _off(got, want):
    return float(np.sqrt(np.mean(np.square(got - want)) / np.mean(np.square(want))))


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("k", [736, 768 + 32, 1024 - 64, 1024 + 64, 4096 + 192, 16384 - 128, 16384 + 64])
def test_products(ctx, qtype, k):
    n = 300
    rng = np.random.default_rng(k + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    w = o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64)
    qt = q.QuantizedTensor([n, k], qtype, packed)
    dw = q.DeviceWeight.upload(qt, ctx)
    assert np.array_equal(dw.download().data, packed)
    bias = rng.standard_normal(n).astype(np.float32)
    for rows in (1, 2, 7, 8, 9, 10, 16, 17, 39, 40, 65, 130):
        x = rng.standard_normal((rows, k)).astype(np.float32)
        got = q.quantized_matmul(x, dw, bias, ctx)
        assert _off(got, x.astype(np.float64) @ w.T + bias) <= 3e-7 + 2.0 ** -22 * 2 ** 0.5, rows
    if k % 64 == 0:
        for rows in (1, 24, 100, 300):
            bits = q.f32_to_bf16_bits(rng.standard_normal((rows, k)).astype(np.float32))
            got = q.quantized_matmul_bf16(bits, dw, ctx)
            assert _off(got, q.bf16_bits_to_f32(bits).astype(np.float64) @ w.T) <= 3e-7, rows
    dw.free()


@pytest.mark.parametrize("qtype", TYPES)
def test_large_elements_in_the_last_block(ctx, qtype):
    """The block in front of the zeros holds the row's largest elements, and bf16 rows take the large tiles."""
    n, k, rows = 1500, 1024 + 32 * 2, 600
    rng = np.random.default_rng(qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    w = o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64)
    qt = q.QuantizedTensor([n, k], qtype, packed)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[:, -32:] *= 1000
    bits = q.f32_to_bf16_bits(x)
    assert _off(q.quantized_matmul_bf16(bits, qt, ctx), q.bf16_bits_to_f32(bits).astype(np.float64) @ w.T) <= 4e-7
    assert _off(q.quantized_matmul(x[:20], qt, None, ctx), x[:20].astype(np.float64) @ w.T) <= 4e-7


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("n,k", [(1, 800), (70, 832), (300, 1088), (129, 2240), (129, 2336)])
def test_rows_end_where_they_end(ctx, qtype, n, k):
    """What lies behind a row's last block is the next row, whose weights may be anything, and behind the last row nothing."""
    rng = np.random.default_rng(n + k + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k)).reshape(n, k // 32, -1).copy()
    odd = np.arange(n) % 2 == 1
    packed[odd] = rng.integers(0, 256, size=packed[odd].shape, dtype=np.uint8)  # scales with infinities and NaN among them, codes of every value
    packed[odd, :8, :2] = np.array([np.inf], np.float16).view(np.uint8)
    w = o.dequantize(qtype, packed.reshape(-1), n * k).reshape(n, k).astype(np.float64)[~odd]
    qt = q.QuantizedTensor([n, k], qtype, packed.reshape(-1))
    for rows in (1, 3, 8, 13, 40, 130):
        x = rng.standard_normal((rows, k)).astype(np.float32)
        got = q.quantized_matmul(x, qt, None, ctx)[:, ~odd]
        assert _off(got, x.astype(np.float64) @ w.T) <= 3e-7 + 2.0 ** -22 * 2 ** 0.5, rows
        if k % 64 == 0:
            bits = q.f32_to_bf16_bits(x)
            got = q.quantized_matmul_bf16(bits, qt, ctx)[:, ~odd]
            assert _off(got, q.bf16_bits_to_f32(bits).astype(np.float64) @ w.T) <= 3e-7, rows


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("k", [736, 992, 1760, 4064, 4128])
def test_the_gemm_takes_multiples_of_64(ctx, qtype, k):
    """bf16 rows of another K are refused, whatever the planes hold; f32 rows of it are not."""
    packed = o.quantize(qtype, gen_weight(np.random.default_rng(k), 40, k))
    qt = q.QuantizedTensor([40, k], qtype, packed)
    x = np.random.default_rng(k + 1).standard_normal((9, k)).astype(np.float32)
    for rows in (1, 9):
        with pytest.raises(Exception, match="64"):
            q.quantized_matmul_bf16(q.f32_to_bf16_bits(x[:rows]), qt, ctx)
    want = x.astype(np.float64) @ o.dequantize(qtype, packed, 40 * k).reshape(40, k).astype(np.float64).T
    assert _off(q.quantized_matmul(x, qt, None, ctx), want) <= 3e-7


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("n,k", [(65536, 800), (32768, 2336)])
def test_memory(ctx, qtype, n, k):
    """800 columns: zeros for the scales (2 or 4 bytes of a block) and fifth bits (4) of seven blocks; 2336: for seven whole blocks of 73.  Blocks of memory are 2 MiB."""
    image = np.zeros(o.packed_bytes(qtype, n * k), np.uint8)
    qt = q.QuantizedTensor([n, k], qtype, image)
    q.DeviceWeight.upload(qt, ctx).free()  # what an upload takes beside the weight is there
    ctx.synchronize()
    free = torch.cuda.mem_get_info()[0]
    dw = q.DeviceWeight.upload(qt, ctx)
    ctx.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    dw.free()
    sides = {o.Q4_0: 2, o.Q4_1: 4, o.Q5_0: 6, o.Q5_1: 8, o.Q8_0: 2}[qtype]
    assert used <= image.size + n * 7 * (sides if k == 800 else image.size // (n * k // 32)) + (4 << 20)
