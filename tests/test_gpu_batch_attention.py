"""Attention of many rows at once (more workgroups than the GPU holds of the large ones): every head size, short and ragged contexts,
grouped heads and a sliding window, against the CPU decode oracle: greedy ids identical, logits within 1e-3 of their range, as for
the one-sequence step."""
import numpy as np
import pytest

import oracle as o
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim,heads,kv,n_seq,window", [(32, 32, 8, 20, None), (64, 16, 16, 40, None), (128, 16, 2, 33, 9), (256, 16, 4, 34, None)])
def test_heads_of_many_sequences(ctx, head_dim, heads, kv, n_seq, window):
    over = dict(num_heads=heads, num_kv_heads=kv, head_dim=head_dim, num_layers=1, max_seq_len=320)
    if window:
        over["sliding_window"] = window
    c = tiny_config(**over)
    w = random_weights(c, head_dim + n_seq, qtype=o.Q8_0)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    rng = np.random.default_rng(n_seq)
    lengths = [[1, 63, 64, 65, 200, 15, 128, 31][i % 8] for i in range(n_seq)]  # a pass of the kernel is 256 / (head_dim / 8) positions
    prompts = [rng.integers(0, c["vocab_size"], size=n) for n in lengths]
    got, _, _ = gpu.generate_batch(prompts, 3)
    for s in range(8):
        nxt = None
        for pos, t in enumerate(prompts[s]):
            nxt, _ = cpu.forward(int(t), pos)
        for i in range(3):
            assert got[s, i] == nxt, (s, i)
            nxt, lg = cpu.forward(int(nxt), lengths[s] + i)
    _, logits = gpu.forward_batch(got[:, -1].tolist())  # of the next tokens: sequence 7 is the last the oracle walked
    assert max_rel_err(logits[7], lg, DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()
