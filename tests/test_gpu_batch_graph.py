"""Steps of many sequences become a graph once some have been plain launches: every step against the oracle, through the capture, behind a product that
moves the GEMM's scratch from under the graph, and where there is no room for it."""
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
