"""Batched steps of up to eight sequences: gate and up leave the operands of the down projection, where their rows fill the chip without K in parts."""
import numpy as np
import pytest

import oracle as o
from tests.decode_common import load_gpu, load_oracle, random_weights, requantize, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gate,down", [(o.Q4_K, o.Q4_K), (o.Q4_K, o.Q4_0), (o.Q5_K, o.Q6_K), (o.Q6_K, o.Q4_1), (o.Q8_0, o.Q8_0), (o.Q5_1, o.Q5_0), (o.Q4_0, o.Q4_K)])
@pytest.mark.parametrize("n_seq,hidden,inter", [(2, 256, 2304), (5, 256, 2304), (8, 256, 2304), (8, 512, 2304), (5, 768, 2304), (8, 1280, 2304), (8, 256, 2048)],
                         ids=["one chunk", "one chunk, five", "one chunk, eight", "two chunks", "three chunks", "five chunks", "too few rows"])
def test_steps_of_several_sequences(ctx, gate, down, n_seq, hidden, inter):
    c = tiny_config(hidden_size=hidden, intermediate_size=inter, num_layers=2, max_seq_len=16)
    w = random_weights(c, n_seq, gate, std=0.03)
    w = requantize(c, w, {(l, "down"): down for l in range(2)}, 7)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    rng = np.random.default_rng([n_seq, hidden])
    steps = rng.integers(0, c["vocab_size"], size=(3, n_seq))
    got = [gpu.forward_batch(t)[1] for t in steps]
    for s in range(n_seq):
        for i in range(3):
            _, lg = cpu.forward(int(steps[i, s]), i)
            assert max_rel_err(got[i][s], lg, DECODE_FLOOR) <= DECODE_RTOL, (s, i)
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("n_tokens", [6, 9])
@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q4_0, o.Q8_0])
def test_rows_of_a_short_prompt(ctx, qtype, n_tokens):
    """Five and eight rows of one chunk, whose first layer's activations the second layer's keys and values are made of."""
    c = tiny_config(intermediate_size=2304, num_layers=2, max_seq_len=16)
    w = random_weights(c, n_tokens, qtype)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(n_tokens).integers(0, c["vocab_size"], size=n_tokens)
    for pos, t in enumerate(tokens):
        _, lg = cpu.forward(int(t), pos)
    _, logits = gpu.forward_tokens(tokens)
    assert max_rel_err(logits, lg, DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("gate,hidden,inter", [(o.Q8_0, 8448, 4352), (o.Q8_0, 16384, 4352), (o.Q6_K, 4096, 4352), (o.Q6_K, 4352, 8448), (o.Q6_K, 4352, 4352),
                                               (o.Q5_K, 12288, 4352), (o.Q5_K, 12544, 4352), (o.Q4_K, 1024, 8448), (o.Q4_K, 1280, 8448)])
def test_long_rows_and_uneven_rounds(ctx, gate, hidden, inter):
    """Rows of 33 chunks and of the most there are, and either side of each line between a launch that leaves operands and one of their own."""
    c = tiny_config(hidden_size=hidden, intermediate_size=inter, num_layers=1, vocab_size=64, max_seq_len=16)
    rng = np.random.default_rng(hidden)
    w = random_weights(dict(c, intermediate_size=256), hidden, gate, std=0.01)
    L = w["layers"][0]
    for name, n, k in (("gate", inter, hidden), ("up", inter, hidden), ("down", hidden, inter)):  # few different rows: the model is large
        L[name] = o.quantize(gate, (rng.standard_normal((251, k)) * 0.01).astype(np.float32)).reshape(251, -1)[np.arange(n) % 251].reshape(-1)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(8)
    steps = rng.integers(0, c["vocab_size"], size=(2, 8))
    got = [gpu.forward_batch(t)[1] for t in steps]
    for s in (0, 7):
        for i in range(2):
            _, lg = cpu.forward(int(steps[i, s]), i)
            assert max_rel_err(got[i][s], lg, DECODE_FLOOR) <= DECODE_RTOL, (s, i)
    gpu.close()
    cpu.close()
