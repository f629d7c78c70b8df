"""A prompt whose last token goes beside the rows through one layer, which is the first and the last: logits, keys and values as with the step behind the rows."""
import numpy as np
import pytest

from tests.decode_common import load_gpu, random_weights, tiny_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("n_tokens", [12, 65, 200])
def test_step_on_two_streams(ctx, monkeypatch, layers, n_tokens):
    c = tiny_config(max_seq_len=220, num_layers=layers)
    w = random_weights(c, n_tokens)
    beside, behind = load_gpu(ctx, c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(n_tokens).integers(0, c["vocab_size"], size=n_tokens)
    for _ in range(2):
        monkeypatch.setenv("AXQ_STEP_BESIDE", "1")
        got = beside.forward_tokens(tokens)
        monkeypatch.setenv("AXQ_STEP_BESIDE", "0")
        want = behind.forward_tokens(tokens)
        assert got[0] == want[0] and np.array_equal(got[1], want[1])
        for which in (0, 1):
            assert np.array_equal(beside.kv(layers - 1, which)[:, :n_tokens], behind.kv(layers - 1, which)[:, :n_tokens])
        got, want = beside.forward(int(got[0])), behind.forward(int(want[0]))
        assert got[0] == want[0] and np.array_equal(got[1], want[1])
        beside.reset()
        behind.reset()
    beside.close()
    behind.close()
