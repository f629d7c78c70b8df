"""Attention of more heads times sequences than the GPU holds as workgroups of 512 threads: two query heads to 256 threads.  Positions around a pass of such a
workgroup and around the passes it has under way, an odd head left over in a group, a window, against the CPU decode oracle."""
import numpy as np
import pytest

import oracle as o
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim,heads,kv,n_seq,window", [(32, 32, 8, 33, 0), (64, 24, 8, 64, 0), (128, 24, 8, 44, 70), (128, 20, 4, 64, 0), (256, 18, 6, 58, 0)])
def test_two_heads_to_a_small_workgroup(ctx, head_dim, heads, kv, n_seq, window):
    c = tiny_config(num_heads=heads, num_kv_heads=kv, head_dim=head_dim, num_layers=1, max_seq_len=300, sliding_window=window)
    w = random_weights(c, head_dim + n_seq, qtype=o.Q8_0)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    rng = np.random.default_rng(n_seq)
    per_pass = 4 * 64 // (head_dim // 8)  # positions of a pass of four waves, of which four are under way together
    lengths = [[1, per_pass - 1, per_pass, per_pass + 1, 4 * per_pass, 4 * per_pass + 1, 2][i % 7] for i in range(n_seq)]
    prompts = [rng.integers(0, c["vocab_size"], size=n) for n in lengths]
    got, _, _ = gpu.generate_batch(prompts, 2)
    _, logits = gpu.forward_batch(got[:, -1].tolist())
    for s in [*range(7), n_seq - 1]:
        nxt = None
        for pos, t in enumerate(prompts[s]):
            nxt, _ = cpu.forward(int(t), pos)
        for i in range(2):
            assert got[s, i] == nxt, (s, i)
            nxt, lg = cpu.forward(int(nxt), lengths[s] + i)
        assert max_rel_err(logits[s], lg, DECODE_FLOOR) <= DECODE_RTOL, s
    gpu.close()
    cpu.close()
