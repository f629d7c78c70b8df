"""The logits of a prompt come from the step of its last token, behind the rows of the others; described layers take that step beside the last
rows: both sides of every edge."""
import numpy as np
import pytest

import oracle as o

from . import gemosun_common as gc
from . import lakulix_common as lc
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tokens", [1, 2, 8, 9, 10, 11, 32, 33, 34, 65])
def test_last_token_of_a_prompt(ctx, monkeypatch, n_tokens):
    monkeypatch.setenv("AXQ_PROMPT_CHUNK", "32")
    c = tiny_config(max_seq_len=80)
    w = random_weights(c, n_tokens)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(n_tokens).integers(0, c["vocab_size"], size=n_tokens)
    for pos, t in enumerate(tokens):
        want, lg = cpu.forward(int(t), pos)
    for fresh in (True, False):
        got, logits = gpu.forward_tokens(tokens)
        assert got == want and max_rel_err(logits, lg, DECODE_FLOOR) <= DECODE_RTOL
        assert gpu.seq_len() == n_tokens
        hidden = gpu.hidden()
        gpu.truncate(n_tokens - 1)  # the same token by the step
        again, step = gpu.forward(int(tokens[-1]))
        assert again == want and max_rel_err(logits, step, DECODE_FLOOR) <= DECODE_RTOL
        assert np.abs(gpu.hidden() - hidden).max() <= DECODE_RTOL * np.abs(hidden).max()
        if fresh:
            gpu.reset()
    nxt, lg = cpu.forward(int(want), n_tokens)
    got, logits = gpu.forward(int(want))
    assert got == nxt and max_rel_err(logits, lg, DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("qtype,sizes", [(o.Q4_K, {}), (o.F32, {}), (o.Q8_0, dict(hidden_size=320, intermediate_size=448, num_heads=5, num_kv_heads=1))],
                         ids=["superblocks", "f32 weights", "no whole superblocks"])
@pytest.mark.parametrize("n_tokens", [2, 9, 10, 11, 33, 41, 65, 71])
def test_logits_have_the_bits_of_the_step(ctx, qtype, sizes, n_tokens):
    """The last token of a prompt goes through the layers as the vector that it is, not as a row of a product with fewer bits."""
    c = tiny_config(max_seq_len=80, **sizes)
    gpu = load_gpu(ctx, c, random_weights(c, n_tokens, qtype))
    tokens = np.random.default_rng(n_tokens).integers(0, c["vocab_size"], size=n_tokens)
    got, logits = gpu.forward_tokens(tokens)
    hidden = gpu.hidden()
    gpu.truncate(n_tokens - 1)
    want, step = gpu.forward(int(tokens[-1]))
    assert got == want and np.array_equal(logits, step) and np.array_equal(hidden, gpu.hidden())
    gpu.close()


LAKULIX = lc.config([lc.lightning(), lc.attention(), lc.wkv(), lc.attention()], width=96, vocab=150)
GEMOSUN = gc.config([gc.attention(mlp=gc.dense(56)), gc.attention(heads=6, kv_heads=3, dim=16, size=41, pool=7, mlp=gc.moe()), gc.attention(size=9, pool=3)], vocab=150)


@pytest.mark.parametrize("kind,cfg", [(lc, LAKULIX), (gc, GEMOSUN)], ids=["lakulix", "gemosun"])
@pytest.mark.parametrize("n_tokens", [2, 3, 32, 33, 34, 65, 66])
def test_step_beside_the_last_rows(ctx, monkeypatch, kind, cfg, n_tokens):
    """A prompt leaves the bits of its rows and then the step, whatever the portions, prompt after prompt."""
    monkeypatch.setenv("AXQ_PROMPT_CHUNK", "32")
    t = kind.tensors(cfg, n_tokens)
    beside, apart = kind.product(cfg, t, "bfloat16", ctx, 200), kind.product(cfg, t, "bfloat16", ctx, 200)
    for start in range(3):
        tokens = np.random.default_rng([n_tokens, start]).integers(0, cfg["vocab"], size=n_tokens)
        got, logits = beside.forward_tokens(tokens)
        apart.forward_rows(tokens[:-1])
        want, lg = apart.forward(int(tokens[-1]))
        assert got == want and np.array_equal(logits, lg)
        assert np.array_equal(beside.hidden(), apart.hidden()) and beside.seq_len() == apart.seq_len()
        if start == 1:
            beside.reset()
            apart.reset()
    beside.close()
    apart.close()
