"""GPU parity of the step's attention with one workgroup per group of query heads: contexts at the edges of its passes over the cache (head sizes
32 to 256 take 128 to 16 positions at a time, four times that on one trip), one and two query heads to a workgroup, an odd number
of them per KV head, a sliding window that starts inside a pass, the first position of an empty cache."""
import numpy as np
import pytest

import oracle as o
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,head_dim,heads,kv,window,lengths", [
    (1, 128, 4, 2, 0, (0, 1, 31, 32, 127, 128, 129, 600)),
    (1, 256, 2, 1, 0, (15, 16, 17, 64, 65)),
    (1, 32, 8, 2, 0, (127, 511, 512, 513)),
    (64, 128, 4, 2, 0, (0, 128, 131)),          # 256 query heads: two to a workgroup
    (64, 128, 6, 2, 0, (33, 130)),              # three per KV head: the second workgroup has one
    (64, 64, 8, 2, 0, (255, 256)),
    (33, 32, 8, 1, 0, (127, 129)),
    (48, 256, 8, 2, 0, (16, 65)),
    (64, 128, 4, 2, 37, (36, 37, 150)),
    (1, 128, 4, 2, 130, (129, 130, 300)),
    (1, 256, 2, 2, 0, (319, 320, 321)),         # where one sequence's positions are split
    (1, 256, 4, 1, 0, (511, 512, 513)),
    (1, 128, 4, 2, 0, (639, 640, 641)),
    (3, 256, 2, 2, 0, (320, 639, 640, 641)),
])
def test_step_attention_at_the_edges_of_its_passes(ctx, n_seq, head_dim, heads, kv, window, lengths):
    c = tiny_config(max_seq_len=max(lengths) + 8, num_heads=heads, num_kv_heads=kv, head_dim=head_dim, sliding_window=window)
    w = random_weights(c, 500 + head_dim + n_seq)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    rng = np.random.default_rng(head_dim + n_seq)
    prompt = rng.integers(0, c["vocab_size"], size=max(lengths) + 1).astype(np.int32)
    for pos, t in enumerate(prompt):
        if pos in lengths:
            gpu.reset()
            if pos:
                gpu.forward_tokens(prompt[:pos], want_logits=False)
            for s in range(1, n_seq):
                gpu.copy_sequence(0, s)
            toks = np.resize([t, (int(t) + 1) % c["vocab_size"]], n_seq)  # neighbours differ
            got = gpu.forward_batch(toks)[1]
            other = cpu.forward(int(toks[-1]), pos)[1]
            want = cpu.forward(int(t), pos)[1]
            assert max_rel_err(got[0], want, DECODE_FLOOR) <= DECODE_RTOL, pos
            assert max_rel_err(got[-1], other if n_seq % 2 == 0 else want, DECODE_FLOOR) <= DECODE_RTOL, pos
        else:
            cpu.forward(int(t), pos)
    gpu.close()
    cpu.close()
