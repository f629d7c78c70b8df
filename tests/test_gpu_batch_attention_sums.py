"""Batched steps whose q, k and v reach the attention as sums of parts of K: fewer parts than the eight it requests at once (2, 4, 3, 4), as many, and more
(9, 11, 16), rows as limbs and as pairs, one and two heads to a workgroup, against the CPU decode oracle."""
import numpy as np
import pytest

import oracle as o
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,n_seq,head_dim,heads,kv,qtype", [(512, 44, 64, 8, 2, o.Q4_K), (1024, 64, 128, 24, 8, o.Q5_K), (1536, 10, 32, 4, 4, o.Q8_0), (2048, 12, 128, 6, 2, o.Q4_K),
                                                                 (2048, 50, 64, 12, 3, o.Q6_K), (2048, 33, 256, 10, 2, o.Q4_0),
                                                                 (2304, 39, 64, 16, 8, o.Q8_0), (2816, 34, 128, 8, 4, o.Q6_K), (4096, 35, 128, 8, 4, o.Q4_K)])
def test_steps_over_parts_of_k(ctx, hidden, n_seq, head_dim, heads, kv, qtype):
    c = tiny_config(hidden_size=hidden, num_heads=heads, num_kv_heads=kv, head_dim=head_dim, num_layers=2, max_seq_len=16)
    w = random_weights(c, n_seq, qtype, std=0.03)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    steps = np.random.default_rng([n_seq, hidden]).integers(0, c["vocab_size"], size=(3, n_seq))
    got = [gpu.forward_batch(t)[1] for t in steps]
    for s in (0, 1, n_seq // 2, n_seq - 1):
        for i in range(3):
            _, lg = cpu.forward(int(steps[i, s]), i)
            assert max_rel_err(got[i][s], lg, DECODE_FLOOR) <= DECODE_RTOL, (s, i)
    gpu.close()
    cpu.close()
