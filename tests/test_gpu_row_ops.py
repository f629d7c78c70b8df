"""Row operations of a prompt's described layers in steps of four columns: rows that end inside a step, rows wider than what a
workgroup keeps in registers (4096 and 8192 columns), gate groups of a power of two, of any other size and of the whole row."""
import numpy as np
import pytest

from . import lakulix_common as lc
from .stack_common import close, feed, tokens_of

pytestmark = pytest.mark.gpu
CASES = {
    "group 4": (lc.config([lc.wkv(heads=3, dim=4)], width=41), {}),
    "group 16": (lc.config([lc.wkv(heads=5, dim=16)], width=66), {}),
    "group 256": (lc.config([lc.wkv(heads=2, dim=256)], width=64), {}),
    "groups beyond 1024": (lc.config([lc.wkv(heads=65, dim=32)], width=1027), {}),
    "group 100": (lc.config([lc.wkv(heads=3, dim=100)], width=64), {}),
    "row of 300": (lc.config([lc.lightning(heads=3, dim=16, vdim=100)], width=1026), {}),
    "row of 4104": (lc.config([lc.lightning(heads=27, dim=4, vdim=152)], width=70), {}),
    "row of 8197": (lc.config([lc.lightning(heads=1, dim=8, vdim=8, ff=8197)], width=40), {}),
    "row of 9000": (lc.config([lc.lightning(heads=1, dim=8, vdim=8, ff=9000)], width=40), {}),
}


@pytest.mark.parametrize("dtype", ("float32", "bfloat16"))
@pytest.mark.parametrize("name", sorted(CASES))
def test_rows(ctx, name, dtype):
    cfg, kw = CASES[name]
    t = lc.tensors(cfg, 17, **kw)
    tokens = tokens_of(cfg, 37)
    want, runs = lc.oracle(cfg, t).forward(tokens)
    m = lc.product(cfg, t, dtype, ctx)
    got, layers = m.forward_rows(tokens, range(len(tokens)), layers=True)
    assert np.abs(layers - runs).max() <= lc.LIMIT[dtype] * np.abs(runs).max() # the bound of the layers' own tests
    assert close(got, want, dtype)
    m.close()


STATES = {
    "64 by 36": lc.config([lc.lightning(heads=2, dim=64, vdim=36)], width=64),
    "52 by 32": lc.config([lc.lightning(heads=1, dim=52, vdim=32)], width=64),
    "128 by 100": lc.config([lc.lightning(heads=2, dim=128, vdim=100)], width=64),
    "per token 64": lc.config([lc.wkv(heads=3, dim=64)], width=64),
    "per token 100": lc.config([lc.wkv(heads=1, dim=100)], width=64),
}


@pytest.mark.parametrize("name", sorted(STATES))
def test_two_columns_of_a_state(ctx, name):
    """Key and value sizes that take two columns of a state per lane, in portions of one segment, several and a part of one."""
    cfg = STATES[name]
    t = lc.tensors(cfg, 23)
    tokens = tokens_of(cfg, 330)
    want = lc.oracle(cfg, t).forward(tokens)[0]
    m = lc.product(cfg, t, "float32", ctx)
    assert close(feed(m, tokens, [17, 290, 22, 1]), want, "float32")
    m.close()
