"""What stands at the ends of a one-token step: the splits of its attention put together, at every count where the merge takes another way
(8 values of a wave ahead, 32 splits, 64 to a lane each), and the last of several largest logits."""
import numpy as np
import pytest

from . import gemosun_common as gc
from . import lakulix_common as lc
from .stack_common import close, feed
from .test_gpu_gemosun import _pointing_model as soft_model, one
from .test_gpu_lakulix import _pointing_model as sigmoid_model

pytestmark = pytest.mark.gpu


def _check(ctx, product, oracle, cfg, t, places, dtype="bfloat16"):
    n = places[-1] + 3
    tokens = np.random.default_rng(8).integers(3, cfg["vocab"], n)
    tokens[7] = 2
    cuts, at = [], 0
    for p in places: # rows up to there, then three steps, of which the second asks for the token far back
        cuts += [p - at, 1, 1, 1]
        at = p + 3
        tokens[p + 1] = 1
    want = oracle(cfg, t).forward(tokens)[0]
    m = product(cfg, t, dtype, ctx, n + 5)
    assert close(feed(m, tokens, cuts), want, dtype) # the bound of the layers' own tests
    m.close()


@pytest.mark.parametrize("size,pool", [(4300, 64), (33, 1), (2100, 3)])
def test_softmax_splits(ctx, size, pool):
    cfg, t = soft_model(64, size, pool)
    _check(ctx, gc.product, gc.oracle, cfg, t, (63, 2046, 2110, 4094, 4158))


def test_sigmoid_splits(ctx):
    cfg, t = sigmoid_model(32, 48, 16, 128, 4300)
    _check(ctx, lc.product, lc.oracle, cfg, t, (63, 510, 2046, 2110, 2300))


@pytest.mark.parametrize("vocab", [101, 1024, 4099, 33003])
def test_last_of_the_largest(ctx, vocab):
    cfg = one(heads=1, kv_heads=1, dim=16, width=32, vocab=vocab)
    t = gc.tensors(cfg, 3)
    m = gc.product(cfg, t, "float32", ctx)
    got = m.forward(5)
    top, first = int(np.argmax(got[1])), int(got[0])
    m.close()
    assert top == first
    for others in ((7, vocab - 1), (0, 8), (vocab // 2, vocab // 2 + 1)):
        u = dict(t)
        u["head"] = t["head"].copy()
        u["head"][list(others)] = t["head"][top]
        m = gc.product(cfg, u, "float32", ctx)
        nxt, logits = m.forward(5)
        equal = np.flatnonzero(logits == logits.max())
        m.close()
        assert set(others) | {top} == set(equal.tolist()) and int(nxt) == equal[-1]
