"""What steps and prompts hand over: logits that come to the caller's memory by portions, at the edges of a portion, and memory that a program may
keep and that the processes it forks have."""
import numpy as np
import pytest

from . import lakulix_common as lc
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


def _stays_behind(a):
    """Whether a forked process lacks the pages of an array (`dc`: do not copy on fork)."""
    here, at = False, a.ctypes.data
    with open("/proc/self/smaps") as f:
        for line in f:
            head = line.split()[0]
            if not head.endswith(":"):
                lo, hi = (int(v, 16) for v in head.split("-"))
                here = lo <= at < hi
            elif here and head == "VmFlags:":
                return "dc" in line.split()
    raise AssertionError("no such mapping")


def test_results_are_kept_and_forked(ctx):
    c = tiny_config(vocab_size=32000)
    gpu = load_gpu(ctx, c, random_weights(c, 5))
    kept = [gpu.forward_tokens([1, 2, 3])[1]] + [gpu.forward(t)[1] for t in range(40)]
    copies = [k.copy() for k in kept]
    gpu.truncate(0)
    again = [gpu.forward_tokens([1, 2, 3])[1]] + [gpu.forward(t)[1] for t in range(40)]
    gpu.set_batch(2)
    kept.append(gpu.forward_batch([1, 2])[1])
    assert all(np.array_equal(a, b) and np.array_equal(a, d) for a, b, d in zip(kept, copies, again))
    assert not any(_stays_behind(a) for a in kept)
    gpu.close()


@pytest.mark.parametrize("n_seq,vocab", [(1, 262144), (1, 262148), (3, 87384), (32, 16384), (64, 8196), (64, 18724)])
def test_logits_come_by_portions(ctx, n_seq, vocab):
    """One portion of a megabyte, a few bytes more, two, two and a few bytes, five."""
    c = tiny_config(vocab_size=vocab, num_layers=1)
    w = random_weights(c, vocab)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(n_seq).integers(0, vocab, size=n_seq)
    if n_seq > 1:
        gpu.set_batch(n_seq)
        nxt, logits = gpu.forward_batch(tokens)
    else:
        t, logits = gpu.forward(int(tokens[0]))
        nxt, logits = [t], logits.reshape(1, -1)
    for s in range(n_seq):
        want, lg = cpu.forward(int(tokens[s]), 0)
        assert nxt[s] == want and max_rel_err(logits[s], lg, DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()


def test_layer_outputs_go_to_the_call_that_wants_them(ctx, monkeypatch):
    """A call that fails leaves no place behind where a later prompt would write its layers' outputs."""
    cfg = lc.config([lc.attention(), lc.lightning()], width=96, vocab=150)
    m = lc.product(cfg, lc.tensors(cfg, 3), "bfloat16", ctx)
    tokens = np.arange(20, dtype=np.int32)
    layers, logits = np.full((2, 20, 96), 7, np.float32), np.full((1, 150), 7, np.float32)
    place = np.array([19], np.int32)
    call = lambda: m.ctx.lib.axq_model_forward_rows(m.handle, tokens.ctypes.data, 20, place.ctypes.data, 1, logits.ctypes.data, layers.ctypes.data)  # noqa: E731
    monkeypatch.setenv("AXQ_GEMM_SCRATCH_MAX", "0")
    assert call() != 0
    monkeypatch.delenv("AXQ_GEMM_SCRATCH_MAX")
    got = m.forward_tokens(tokens)[1]
    m.reset()
    m.forward_rows(tokens, [3])
    assert (layers == 7).all() and (logits == 7).all()
    m.reset()
    assert call() == 0 and not (layers == 7).any() and not (logits == 7).any()
    assert np.abs(logits[0] - got).max() <= lc.LIMIT["bfloat16"] * np.abs(got).max()
    m.close()
