"""Forked sequences hold what the first one holds, around the pieces that a workgroup of the copy takes: steps behind the fork are the same for all, bit for bit."""
import numpy as np
import pytest

from tests.decode_common import load_gpu, random_weights, tiny_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 129])
def test_forks_step_alike(ctx, head_dim, n):
    c = tiny_config(max_seq_len=140, head_dim=head_dim)
    gpu = load_gpu(ctx, c, random_weights(c, n))
    gpu.set_batch(3)
    nxt, _ = gpu.forward_tokens(np.random.default_rng(n).integers(0, c["vocab_size"], size=n))
    for s in (1, 2):
        gpu.copy_sequence(0, s)
    for _ in range(3):
        ids, logits = gpu.forward_batch([int(nxt)] * 3)
        assert np.isfinite(logits).all() and np.array_equal(logits[0], logits[1]) and np.array_equal(logits[0], logits[2])
        nxt = ids[0]
    gpu.close()
