"""A prompt that finds no room for its rows takes the model's rows with it: the batched steps behind it reserve rows of their own, in front of any
graph, and give the right results or say that there is no room; with room again they go on."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,qtype", [(2, o.Q4_K), (8, o.Q8_0), (12, o.Q4_K), (64, o.Q5_1)])
@pytest.mark.parametrize("room", [0, 8])
@pytest.mark.parametrize("tokens", [20, 100])
def test_steps_behind_a_prompt_without_room(monkeypatch, n_seq, qtype, room, tokens):
    ctx = q.Context(0)
    c = tiny_config(max_seq_len=160)
    w = random_weights(c, 700 + n_seq, qtype=qtype)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    gpu.set_batch(n_seq)
    rng = np.random.default_rng(n_seq)
    tok, pos = int(rng.integers(0, c["vocab_size"])), 0

    def step():  # all sequences feed the same; the last one is never anything else
        nonlocal tok, pos
        got_next, got = gpu.forward_batch(np.full(n_seq, tok))
        want_next, want = cpu.forward(tok, pos)
        assert got_next[-1] == want_next and max_rel_err(got[-1], want, DECODE_FLOOR) <= DECODE_RTOL, pos
        tok, pos = int(want_next), pos + 1

    for _ in range(11):  # plain launches, then graph launches
        step()
    monkeypatch.setenv("AXQ_PROMPT_ROWS_MAX", str(room))
    try:
        gpu.forward_tokens(rng.integers(0, c["vocab_size"], size=tokens))
    except Exception as e:
        assert "activations for" in str(e)
    for _ in range(2):
        try:
            step()
        except AssertionError:
            raise
        except Exception as e:
            assert "activations for" in str(e) and (room == 0 or n_seq > 32)
    monkeypatch.delenv("AXQ_PROMPT_ROWS_MAX")
    for _ in range(11):
        step()
    gpu.close()
    cpu.close()
    ctx.close()
