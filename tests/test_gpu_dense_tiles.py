"""The tiles of the products with bfloat16 weights, through models whose one wide product takes them: row and column counts on both
sides of their edges, odd steps for two groups of waves, K beyond the stages in LDS, columns whose rows are no whole 16 bytes, a few narrow weights beside a
wide one, and what happens to a result on its way out (softcap, GLU, residual, the mean over the layers)."""
import pytest

from . import gemosun_common as gc
from . import lakulix_common as lc
from .stack_common import close, feed, tokens_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,vocab,width", [(300, 22003, 64), (257, 22004, 200), (129, 17000, 72), (150, 8300, 192), (140, 8301, 64), (200, 4400, 130),
                                              (70, 300, 320), (300, 22003, 1600), (257, 17004, 1544), (260, 17000, 1536),
                                              (150, 8300, 384), (150, 8300, 704), (140, 8301, 1000), (129, 8200, 1408)])
def test_logits_of_every_tile(ctx, rows, vocab, width):
    cfg = lc.config([lc.wkv(heads=2, dim=8)], width=width, vocab=vocab)
    t = lc.tensors(cfg, rows + width)
    tokens = tokens_of(cfg, rows)
    want = lc.oracle(cfg, t).forward(tokens)[0]
    m = lc.product(cfg, t, "bfloat16", ctx)
    assert close(m.forward_rows(tokens, range(rows)), want, "bfloat16")
    m.close()


@pytest.mark.parametrize("rows,ff", [(300, 11000), (270, 10977), (150, 4200)])
def test_wide_feed_forward_beside_narrow_projections(ctx, rows, ff):
    cfg = gc.config([gc.attention(heads=3, kv_heads=1, dim=16, mlp=gc.dense(ff)), gc.attention(mlp=gc.dense(40))], width=96, vocab=150)
    t = gc.tensors(cfg, 5)
    tokens = tokens_of(cfg, rows)
    want = gc.oracle(cfg, t).forward(tokens)[0]
    m = gc.product(cfg, t, "bfloat16", ctx, 400)
    assert close(feed(m, tokens, [rows]), want, "bfloat16", 2)
    m.close()


def test_wide_feed_forward_beside_narrow_projections_of_long_rows(ctx):
    """256 x 256 outputs, which rows of fewer than 1536 elements do not take, and a second launch for the narrow weights."""
    cfg = gc.config([gc.attention(heads=3, kv_heads=1, dim=16, mlp=gc.dense(7000))], width=1544, vocab=150)
    t = gc.tensors(cfg, 6)
    tokens = tokens_of(cfg, 270)
    want = gc.oracle(cfg, t).forward(tokens)[0]
    m = gc.product(cfg, t, "bfloat16", ctx, 400)
    assert close(feed(m, tokens, [270]), want, "bfloat16", 1)
    m.close()
