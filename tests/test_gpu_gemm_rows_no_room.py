"""What ran before the GEMM took it still runs when the card has no room for the GEMM's scratch: calls of 10 to 39 rows, prompts of up
to 31 tokens and steps of 10 to 24 sequences fall back on the small-batch GEMV, which needs none."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, gen_weight, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture
def full_card(monkeypatch):
    """A context whose GEMM scratch cannot be allocated."""
    ctx = q.Context(0)
    monkeypatch.setenv("AXQ_GEMM_SCRATCH_MAX", "0")
    yield ctx
    monkeypatch.delenv("AXQ_GEMM_SCRATCH_MAX")


@pytest.mark.parametrize("qtype,rows", [(o.Q4_K, 10), (o.Q4_0, 21), (o.Q8_0, 39)])
def test_few_rows(full_card, monkeypatch, qtype, rows):
    rng = np.random.default_rng(rows)
    n, k = 300, 1024
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    qt = q.QuantizedTensor([n, k], qtype, packed)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    want = x.astype(np.float64) @ o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64).T
    got = q.quantized_matmul(x, qt, None, full_card)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()  # some 2^-17: sums of 1024 products in f32
    with pytest.raises(Exception, match="AXQ_GEMM_SCRATCH_MAX"):
        q.quantized_matmul(np.tile(x, (8, 1)), qt, None, full_card)  # many rows need it
    monkeypatch.delenv("AXQ_GEMM_SCRATCH_MAX")
    got = q.quantized_matmul(x, qt, None, full_card)  # room again
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    monkeypatch.setenv("AXQ_GEMM_SCRATCH_MAX", "0")


@pytest.mark.parametrize("n_tokens", [12, 20, 32])
def test_prompts(full_card, n_tokens):
    c = tiny_config(max_seq_len=64)
    w = random_weights(c, n_tokens)
    cpu, gpu = load_oracle(c, w), load_gpu(full_card, c, w)
    tokens = np.random.default_rng(n_tokens).integers(0, c["vocab_size"], size=n_tokens)
    for pos, t in enumerate(tokens):
        nxt, lg = cpu.forward(int(t), pos)
    got, logits = gpu.forward_tokens(tokens)
    assert got == nxt and max_rel_err(logits, lg, DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("n_seq", [10, 24])
def test_steps_of_many_sequences(full_card, n_seq):
    c = tiny_config(max_seq_len=64)
    w = random_weights(c, n_seq)
    cpu, gpu = load_oracle(c, w), load_gpu(full_card, c, w)
    gpu.set_batch(n_seq)
    rng = np.random.default_rng(n_seq)
    prompts = [rng.integers(0, c["vocab_size"], size=1 + s % 5) for s in range(n_seq)]
    got, _, _ = gpu.generate_batch(prompts, 4)
    for s, p in enumerate(prompts):
        for pos, t in enumerate(p):
            nxt, _ = cpu.forward(int(t), pos)
        for i in range(4):
            assert got[s, i] == nxt, (s, i)
            nxt, _ = cpu.forward(int(nxt), len(p) + i)
        assert gpu.seq_len_of(s) == len(p) + 3
    gpu.close()
    cpu.close()
