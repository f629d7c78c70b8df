"""Steps of many sequences become a graph once some have been plain launches: every step against the oracle, through the capture, behind a product that
moves the GEMM's scratch from under the graph, and where there is no room for a graph or the scratch would have to grow while it is captured."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,qtype", [(9, o.Q4_K), (12, o.Q5_1), (26, o.Q8_0), (64, o.Q4_K)])
def test_steps_before_and_after_the_graph(n_seq, qtype):
    ctx = q.Context(0)  # whose scratch is as small as the model's prompts leave it
    c = tiny_config(max_seq_len=40)
    w = random_weights(c, 600 + n_seq, qtype=qtype)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    rng = np.random.default_rng(n_seq)
    weight = q.QuantizedTensor([640, 2048], qtype, o.quantize(qtype, rng.standard_normal((640, 2048)).astype(np.float32)))
    toks = np.resize(rng.integers(0, c["vocab_size"], size=7), n_seq)
    for pos in range(24):
        if pos in (12, 18):  # between steps that are graph launches
            q.quantized_matmul(rng.standard_normal((300 * (pos // 6), 2048)).astype(np.float32), weight, None, ctx)
        got_next, got = gpu.forward_batch(toks)
        want_next, want = cpu.forward(int(toks[0]), pos)
        assert got_next[0] == want_next and max_rel_err(got[0], want, DECODE_FLOOR) <= DECODE_RTOL, pos
        same = [s for s in range(n_seq) if s % 7 == 0]
        assert all(np.array_equal(got[s], got[0]) for s in same), pos
        toks = got_next
    gpu.close()
    cpu.close()
    ctx.close()


def _agree(gpu, cpu, n_seq, tok, first, steps):
    for pos in range(first, first + steps):
        got_next, got = gpu.forward_batch(np.full(n_seq, tok))
        want_next, want = cpu.forward(tok, pos)
        assert got_next[0] == want_next and max_rel_err(got[0], want, DECODE_FLOOR) <= DECODE_RTOL, pos
        assert all(np.array_equal(got[s], got[0]) for s in range(n_seq)), pos
        tok = int(want_next)
    return tok


@pytest.mark.parametrize("n_seq", [5, 12, 40])
def test_no_room_for_a_graph(ctx, monkeypatch, n_seq):
    c = tiny_config(max_seq_len=48)
    w = random_weights(c, n_seq)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    monkeypatch.setenv("AXQ_GRAPH_ROOM", "0")
    tok = _agree(gpu, cpu, n_seq, 3, 0, 20)
    monkeypatch.delenv("AXQ_GRAPH_ROOM")
    _agree(gpu, cpu, n_seq, tok, 20, 20)
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("most", [1 << b for b in range(14, 22)])
def test_scratch_that_would_grow_in_the_capture(monkeypatch, most):
    """The plain launches have less room than they ask for and do with it; the capture asks again, with room now."""
    ctx = q.Context(0)
    c = tiny_config(max_seq_len=48, hidden_size=512, intermediate_size=1024)
    w = random_weights(c, most)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(12)
    monkeypatch.setenv("AXQ_GEMM_SCRATCH_MAX", str(most))
    tok = _agree(gpu, cpu, 12, 3, 0, 8)
    monkeypatch.delenv("AXQ_GEMM_SCRATCH_MAX")
    _agree(gpu, cpu, 12, tok, 8, 12)
    gpu.close()
    cpu.close()
    ctx.close()


@pytest.mark.parametrize("fused", ["0", "14"])
@pytest.mark.parametrize("n_seq", [5, 12, 40])
def test_steps_whose_positions_are_split(ctx, monkeypatch, n_seq, fused):
    """A graph of their own, from the first position on or in the middle of steps that were not."""
    monkeypatch.setenv("AXQ_ATTN_FUSED_MAX", fused)
    c = tiny_config(max_seq_len=48)
    w = random_weights(c, 50 + n_seq)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    _agree(gpu, cpu, n_seq, 3, 0, 40)
    gpu.close()
    cpu.close()
