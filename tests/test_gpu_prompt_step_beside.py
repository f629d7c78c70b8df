"""A prompt's last token goes through the layers beside the rows in front of it: logits, caches, position and what follows against the oracle, prompts in
several chunks, on top of a context, of a batched model, again and again, and where the rows, or the graph of the steps to come, find no room."""
import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.decode_common import load_gpu, load_oracle, random_weights, tiny_config
from tests.util import DECODE_FLOOR, DECODE_RTOL, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def beside(monkeypatch):
    """However small the model."""
    monkeypatch.setenv("AXQ_STEP_BESIDE", "1")


def _walk(cpu, tokens, pos=0):
    for t in tokens:
        nxt, lg = cpu.forward(int(t), pos)
        pos += 1
    return nxt, lg


@pytest.mark.parametrize("lengths", [(193,), (194, 200), (300, 193, 3), (5, 250)])
@pytest.mark.parametrize("chunk", ["2048", "96"])
def test_prompts_on_top_of_each_other(ctx, monkeypatch, lengths, chunk):
    monkeypatch.setenv("AXQ_PROMPT_CHUNK", chunk)
    c = tiny_config(max_seq_len=sum(lengths) + 8, num_layers=3)
    w = random_weights(c, sum(lengths))
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    rng = np.random.default_rng(len(lengths))
    for n_seq in (1, 3):  # with several sequences the first one takes the prompt
        gpu.set_batch(n_seq)
        pos = 0
        for n in lengths:
            tokens = rng.integers(0, c["vocab_size"], size=n)
            want = _walk(cpu, tokens, pos)
            got = gpu.forward_tokens(tokens)
            pos += n
            assert got[0] == want[0] and max_rel_err(got[1], want[1], DECODE_FLOOR) <= DECODE_RTOL, n
        for _ in range(3):  # the steps behind it see its position and its keys
            want, got = cpu.forward(int(want[0]), pos), gpu.forward(int(got[0]))
            pos += 1
            assert got[0] == want[0] and max_rel_err(got[1], want[1], DECODE_FLOOR) <= DECODE_RTOL, pos
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("n", [10, 14, 33])
def test_wide_models(ctx, n):
    c = tiny_config(max_seq_len=n + 4, hidden_size=4096, intermediate_size=512, num_heads=4, num_kv_heads=2, vocab_size=64)
    w = random_weights(c, n)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(n).integers(0, c["vocab_size"], size=n)
    want = _walk(cpu, tokens)
    first = None
    for _ in range(5):  # the same bits every time
        gpu.reset()
        got = gpu.forward_tokens(tokens)
        assert got[0] == want[0] and max_rel_err(got[1], want[1], DECODE_FLOOR) <= DECODE_RTOL
        assert first is None or np.array_equal(first, got[1])
        first = got[1]
    gpu.close()
    cpu.close()


def test_without_room_for_the_rows(monkeypatch):
    ctx = q.Context(0)
    monkeypatch.setenv("AXQ_GEMM_SCRATCH_MAX", "0")
    c = tiny_config(max_seq_len=32, hidden_size=4096, intermediate_size=512, vocab_size=64)
    w = random_weights(c, 9)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(9).integers(0, c["vocab_size"], size=20)
    want = _walk(cpu, tokens)
    for _ in range(2):
        got = gpu.forward_tokens(tokens)  # the rows fail behind the step's first launches and go in by eights
        assert got[0] == want[0] and max_rel_err(got[1], want[1], DECODE_FLOOR) <= DECODE_RTOL
        assert gpu.forward(int(got[0]))[0] == cpu.forward(int(want[0]), 20)[0]
        gpu.reset()
        monkeypatch.delenv("AXQ_GEMM_SCRATCH_MAX", raising=False)
    gpu.close()
    cpu.close()
    ctx.close()


def test_without_room_for_the_graph(ctx, monkeypatch):
    c = tiny_config(max_seq_len=320)
    w = random_weights(c, 11)
    cpu, gpu = load_oracle(c, w), load_gpu(ctx, c, w)
    tokens = np.random.default_rng(11).integers(0, c["vocab_size"], size=300)
    want = _walk(cpu, tokens)
    monkeypatch.setenv("AXQ_GRAPH_ROOM", "0")
    got = gpu.forward_tokens(tokens)  # needs none
    assert got[0] == want[0] and max_rel_err(got[1], want[1], DECODE_FLOOR) <= DECODE_RTOL
    with pytest.raises(Exception, match="AXQ_GRAPH_ROOM"):
        gpu.forward(int(got[0]))  # a step does
    monkeypatch.delenv("AXQ_GRAPH_ROOM")
    want, got = cpu.forward(int(want[0]), 300), gpu.forward(int(got[0]))
    assert got[0] == want[0] and max_rel_err(got[1], want[1], DECODE_FLOOR) <= DECODE_RTOL
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("rows,layers,width", [(191, 2, 1024), (192, 2, 256), (1024, 2, 1024)])
def test_both_sides_of_the_rule(ctx, monkeypatch, rows, layers, width):
    """The same bits beside the rows and behind them, on both sides of where one gives way to the other."""
    c = tiny_config(max_seq_len=rows + 2, num_layers=layers, hidden_size=width, intermediate_size=256, vocab_size=64)
    gpu = load_gpu(ctx, c, random_weights(c, rows))
    tokens = np.random.default_rng(rows).integers(0, c["vocab_size"], size=rows + 1)
    got = []
    for knob in ("0", "1", None):
        monkeypatch.delenv("AXQ_STEP_BESIDE") if knob is None else monkeypatch.setenv("AXQ_STEP_BESIDE", knob)
        gpu.reset()
        got.append(gpu.forward_tokens(tokens)[1])
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    gpu.close()
