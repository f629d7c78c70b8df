"""GPU parity of the tiles whose waves take turns, at the edges of their K: 128 x 128 outputs whose halves have parts of K of their own, even and
uneven, alone and with K split over workgroups; and of operands made with the reduction in front of them or by several workgroups per row."""
import numpy as np
import pytest

import oracle as o
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.test_gpu_gemm_rows import _check
from tests.util import DECODE_FLOOR, DECODE_RTOL, gen_weight, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K])
@pytest.mark.parametrize("rows,n,k,bf16", [
    (40, 129, 2048, False), (64, 127, 2304, False), (41, 1, 2560, False),  # in parts of one superblock, which are too short for it
    (65, 257, 2304, True), (128, 130, 2816, True),
    (48, 8192, 8192, False), (65, 12032, 4608, True),                      # K in four parts of eight and in two of nine
    (130, 2048, 16384, True),                                              # two tiles of rows, eight parts
    (50, 4100, 14336, False)])                                             # seven parts of eight superblocks: the last tile has four columns
def test_halves_with_their_own_k(ctx, qtype, rows, n, k, bf16):
    rng = np.random.default_rng(rows + n + k + qtype)
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    x = rng.standard_normal((rows, k)).astype(np.float32) * (10.0 ** rng.integers(-3, 4, size=(rows, 1))).astype(np.float32)
    _check(ctx, qtype, n, k, packed, x, bias=None if bf16 else rng.standard_normal(n).astype(np.float32), bf16=bf16)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K])
@pytest.mark.parametrize("rows,n,k,bf16", [(40, 16512, 2048, False), (64, 16386, 2304, False), (41, 16385, 2560, False), (65, 16387, 2304, True), (128, 16514, 2816, True)])
def test_halves_with_their_own_k_and_all_of_it(ctx, qtype, rows, n, k, bf16):
    """More tiles than half the compute units, so that K is not split: eight to eleven superblocks."""
    rng = np.random.default_rng(rows + n + k + qtype)
    packed = o.quantize(qtype, gen_weight(rng, 1009, k)).reshape(1009, -1)[np.arange(n) % 1009].reshape(-1)
    x = rng.standard_normal((rows, k)).astype(np.float32) * (10.0 ** rng.integers(-3, 4, size=(rows, 1))).astype(np.float32)
    _check(ctx, qtype, n, k, packed, x, bias=None if bf16 else rng.standard_normal(n).astype(np.float32), bf16=bf16)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K])
@pytest.mark.parametrize("rows,n,k,bf16", [(40, 16385, 256, False), (64, 16386, 512, False), (41, 16387, 768, False), (65, 16512, 1024, True), (128, 16390, 1280, True),
                                           (33, 4096, 1536, True), (50, 513, 4096, False), (64, 6144, 7168, False),
                                           (40, 8192, 1280, False), (64, 12288, 768, False), (66, 8190, 1280, True), (100, 12288, 768, True)])
def test_halves_of_few_superblocks(ctx, qtype, rows, n, k, bf16):
    """One superblock (which shares its K), two, three .. seven, alone and in parts; 33 bf16 rows are no large tile; parts of two of which the last one has
    one, so that its second half has none."""
    rng = np.random.default_rng(rows + n + k + qtype)
    packed = o.quantize(qtype, gen_weight(rng, 509, k)).reshape(509, -1)[np.arange(n) % 509].reshape(-1)
    x = rng.standard_normal((rows, k)).astype(np.float32) * (10.0 ** rng.integers(-3, 4, size=(rows, 1))).astype(np.float32)
    _check(ctx, qtype, n, k, packed, x, bias=None if bf16 else rng.standard_normal(n).astype(np.float32), bf16=bf16)


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q6_K, o.Q8_0])
@pytest.mark.parametrize("rows", [10, 17, 33, 40, 64, 65])
@pytest.mark.parametrize("sizes", [dict(hidden_size=512, intermediate_size=4352, num_heads=8, num_kv_heads=4),
                                   dict(hidden_size=4352, intermediate_size=256, num_heads=4, num_kv_heads=2)], ids=["wide inner", "wide outer"])
def test_operands_made_with_the_reduction(ctx, qtype, rows, sizes):
    """A prompt's rows: the norms and their products behind split products, and SwiGLU over more than 4096 elements."""
    c = tiny_config(max_seq_len=72, vocab_size=64, num_layers=2, **sizes)
    w = random_weights(c, rows, qtype, std=0.02)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(rows).integers(0, c["vocab_size"], size=rows + 1)
    for pos, t in enumerate(tokens):
        want, lg = cpu.forward(int(t), pos)
    got, logits = gpu.forward_tokens(tokens)
    assert max_rel_err(logits, lg, DECODE_FLOOR) <= DECODE_RTOL
    hidden = gpu.hidden()
    gpu.truncate(rows)  # the last token again, by the step
    _, step = gpu.forward(int(tokens[-1]))
    assert np.abs(gpu.hidden() - hidden).max() <= DECODE_RTOL * np.abs(hidden).max()
    assert max_rel_err(logits, step, DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()


def _gate_and_up(ctx, qtype, inter, hidden, rows):
    c = tiny_config(max_seq_len=rows + 8, vocab_size=64, num_layers=2, hidden_size=hidden)  # of a prompt the last layer ends with its keys and values
    w = random_weights(c, rows, qtype, std=0.02)
    c["intermediate_size"] = inter
    rng = np.random.default_rng([rows, inter])
    w["types"] = {}
    for l, L in enumerate(w["layers"]):
        for name, t, shape in (("gate", qtype, (inter, hidden)), ("up", qtype, (inter, hidden)), ("down", o.Q8_0, (hidden, inter))):
            L[name] = o.quantize(t, (rng.standard_normal(shape) * 0.05).astype(np.float32))
            w["types"][(l, name)] = t
    return c, load_oracle(c, w), load_gpu(ctx, c, w), rng


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q6_K, o.Q4_1])
@pytest.mark.parametrize("inter", [8256, 8320], ids=["half a large tile left", "whole tiles"])
@pytest.mark.parametrize("hidden,rows", [(256, 40), (256, 64), (256, 65), (256, 129), (512, 40), (512, 64), (512, 129), (768, 40), (768, 64)])
def test_gate_and_up_leave_their_product(ctx, qtype, inter, hidden, rows):
    """More column tiles than half the compute units, so that a workgroup has all of K: tiles of 256 rows of operands, those of blocks, and tiles of 128, which
    need two superblocks (up to 64 rows of one superblock are activated by the product behind them)."""
    c, cpu, gpu, rng = _gate_and_up(ctx, qtype, inter, hidden, rows)
    tokens = rng.integers(0, c["vocab_size"], size=rows + 1)
    for pos, t in enumerate(tokens):
        _, lg = cpu.forward(int(t), pos)
    _, logits = gpu.forward_tokens(tokens)
    assert max_rel_err(logits, lg, DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K])
@pytest.mark.parametrize("hidden,rows", [(512, 40), (768, 64)])
def test_steps_whose_gate_and_up_leave_their_product(ctx, qtype, hidden, rows):
    c, cpu, gpu, rng = _gate_and_up(ctx, qtype, 8320, hidden, rows)
    gpu.set_batch(rows)
    steps = rng.integers(0, c["vocab_size"], size=(2, rows))
    got = [gpu.forward_batch(t)[1] for t in steps]
    for s in (0, 1, rows // 2, rows - 1):
        for i in range(2):
            _, lg = cpu.forward(int(steps[i, s]), i)
            assert max_rel_err(got[i][s], lg, DECODE_FLOOR) <= DECODE_RTOL, (s, i)
    gpu.close()
    cpu.close()
