"""Nobody reads a prompt's rows behind the last layer's cache or state, so that layer ends there: what it leaves is what rows whose logits are wanted leave."""
import numpy as np
import pytest

from . import gemosun_common as gc
from . import lakulix_common as lc
from .stack_common import LIMIT, error
from tests.decode_common import load_gpu, random_weights, tiny_config

pytestmark = pytest.mark.gpu

LAST = {
    "lightning": (lc, lc.config([lc.attention(ff=40), lc.lightning(ff=56)], width=96, vocab=150)),
    "sigmoid attention": (lc, lc.config([lc.lightning(), lc.attention(heads=6, kv_heads=2, ff=56)], width=96, vocab=150)),
    "wkv": (lc, lc.config([lc.attention(ff=40), lc.wkv(ff=56)], width=96, vocab=150)),
    "alone": (lc, lc.config([lc.attention(ff=40)], width=96, vocab=150)),
    "softmax, dense": (gc, gc.config([gc.attention(mlp=gc.moe()), gc.attention(size=9, pool=3, mlp=gc.dense(56))], vocab=150)),
    "softmax, mixture": (gc, gc.config([gc.attention(mlp=gc.dense(40)), gc.attention(heads=6, kv_heads=3, dim=16, size=41, pool=7, mlp=gc.moe())], vocab=150)),
    "softmax, no feed-forward": (gc, gc.config([gc.attention(mlp=gc.moe()), gc.attention(size=9, pool=3)], vocab=150)),
}


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("name", LAST)
def test_described_layers(ctx, monkeypatch, name, dtype):
    """Two portions, then steps that see what the last layer kept of both.  The products for its cache alone may add up in another order: within what
    every position keeps to against the plain forward."""
    monkeypatch.setenv("AXQ_PROMPT_CHUNK", "32")
    kind, cfg = LAST[name]
    t = kind.tensors(cfg, 3)
    ended, whole = kind.product(cfg, t, dtype, ctx, 100), kind.product(cfg, t, dtype, ctx, 100)
    tokens = np.random.default_rng(4).integers(0, cfg["vocab"], size=54)
    got, want = [ended.forward_tokens(tokens[:50])[1]], []
    whole.forward_rows(tokens[:49])
    want.append(whole.forward(int(tokens[49]))[1])
    for i in tokens[50:]:
        got.append(ended.forward(int(i))[1])
        want.append(whole.forward(int(i))[1])
    assert error(got, want).max() < LIMIT[dtype]
    ended.close()
    whole.close()


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("n_tokens", [2, 9, 32, 49])
def test_llama(ctx, monkeypatch, layers, n_tokens):
    monkeypatch.setenv("AXQ_PROMPT_CHUNK", "32")
    c = tiny_config(max_seq_len=80, num_layers=layers)
    w = random_weights(c, n_tokens)
    ended, whole = load_gpu(ctx, c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(n_tokens).integers(0, c["vocab_size"], size=n_tokens)
    got, logits = ended.forward_tokens(tokens)
    whole.forward_rows(tokens[:-1])
    want, lg = whole.forward(int(tokens[-1]))
    assert got == want and np.array_equal(logits, lg)
    for which in (0, 1):
        assert np.array_equal(ended.kv(layers - 1, which)[:, :n_tokens], whole.kv(layers - 1, which)[:, :n_tokens])
    ended.close()
    whole.close()
