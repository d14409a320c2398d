"""Layers that are alike: one layer's launches made again for the others."""
import ctypes
import shutil
import subprocess

import numpy as np
import pytest
import torch

from alofa_amd.csrc import calls
from alofa_amd.csrc.build import load_binding

SOURCE = """
#include <stdint.h>
static int64_t seen[64];
static int n;
int64_t* places(void) { return seen; }
int keep(int64_t a, float x, int64_t b, int64_t c, float y) { seen[n++] = a, seen[n++] = b, seen[n++] = c, seen[n++] = (int64_t)(x * 2), seen[n++] = (int64_t)(y * 2); return 0; }
void forget(void) { n = 0; }
int odd(int64_t a) { return (int)(a & 1); }
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc") or shutil.which("clang")
    if cc is None:
        pytest.skip("no C compiler")
    d = tmp_path_factory.mktemp("tapes")
    (d / "tapes.c").write_text(SOURCE)
    subprocess.run([cc, "-O2", "-shared", "-fPIC", "-o", str(d / "tapes.so"), str(d / "tapes.c")], check=True)
    return ctypes.CDLL(str(d / "tapes.so"))


@pytest.mark.parametrize("native", [True, False])
def test_calls_are_made_again_with_another_layers_addresses(library, native):
    ways = load_binding() if native else calls
    address = lambda name: ctypes.cast(getattr(library, name), ctypes.c_void_p).value      # noqa: E731
    library.places.restype = ctypes.POINTER(ctypes.c_int64)
    library.forget()
    t = torch.zeros(4)
    assert ways.note(address("keep"), 1, 0.5, 2, 3, 1.5) == 0      # (no tape is being written: a call like any other)
    ways.tape()
    assert ways.note(address("odd"), 7) == 1                       # (a call that failed is not made again)
    assert ways.note(address("keep"), 1000, 2.5, 1099, None, 3.5) == 0
    assert ways.note(address("keep"), 1100, 4.5, 2007, t, -1.5) == 0
    tape = ways.taped((1000, 100), (2000, 8), (5000, 0))
    for at in ((30, 70000, 0), (1 << 40, -5, 1)):
        assert ways.play(tape, at) == 0
    got = np.ctypeslib.as_array(library.places(), (64,))[:40].reshape(8, 5).tolist()
    del tape
    mem = t.data_ptr()
    assert got[:7] == [[1, 2, 3, 1, 3], [1000, 1099, 0, 5, 7], [1100, 2007, mem, 9, -3],
                       [30, 129, 0, 5, 7], [1100, 70007, mem, 9, -3], [1 << 40, (1 << 40) + 99, 0, 5, 7], [1100, 2, mem, 9, -3]]
    with pytest.raises(RuntimeError):
        ways.taped()
    ways.tape()
    ways.note(address("odd"), 8)
    tape = ways.taped((8, 1))
    assert ways.play(tape, (11,)) == 1      # (the first answer that is not zero)
    with pytest.raises(ValueError):
        ways.play(tape, ())


@pytest.mark.parametrize("grows", [False, True])
def test_a_buffer_outgrown_while_a_layer_is_noted(grows):
    """The noted launches before have the old buffer's address: the layers alike run through their parts in that step, and from their notes in the next."""
    from contextlib import contextmanager
    from types import SimpleNamespace as Some
    from alofa_amd.engine.step import StepFunction
    from alofa_amd.model import Model
    ran, played = [], []

    class Block:
        takes_normed, wants_normed, can_leave = True, staticmethod(lambda rows: None), staticmethod(lambda norm: False)

        def forward(self, ctx, i, stream, normed, then):
            ran.append(i)
            ctx.scratch("sums", (8,), torch.float32)
            ctx.scratch("sums", (16 if grows and i else 8,), torch.float32)

    class Tapes:
        sources, source = {1}, {2: 1, 3: 1}

        def stand(self):
            return True

        @contextmanager
        def note(self, i):
            yield Some(play=played.append)

        def addresses(self, i):
            return i
    fn = StepFunction.__new__(StepFunction)
    fn._scratch, fn._views, fn._retired, fn.buffers_moved, fn.device = {}, {}, [], 0, torch.device("cpu")
    fn._eager_scratch = fn._scratch
    model = Model.__new__(Model)
    model.embedding, model.joins, model.streams, model.blocks = Some(forward=lambda ctx, ids: torch.zeros(2, 4)), [], 0, [Block()]
    model.order, model.rt = [Some(layer=0, join=None)] * 5, Some(dtype=torch.float32)
    ctx = Some(fn=fn, scratch=fn.scratch, watch=None, resident=None, tapes=Tapes())
    model.forward(ctx, None)
    assert (ran, played) == (([0, 1, 2, 3, 4], []) if grows else ([0, 1, 4], [2, 3]))
    del ran[:], played[:]
    model.forward(ctx, None)
    assert (ran, played) == ([0, 1, 4], [2, 3])


MODEL = {"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "num_hidden_layers": 7, "hidden_size": 256, "num_attention_heads": 4, "num_key_value_heads": 2, "intermediate_size": 512,
         "vocab_size": 500, "rope_theta": 10000.0, "rms_norm_eps": 1e-6, "tie_word_embeddings": True, "use_sliding_window": False, "max_position_embeddings": 2048}
WINDOWS = {**MODEL, "use_sliding_window": True, "sliding_window": 40, "max_window_layers": 3}


def alike(change=lambda model: None, layers=6):
    """Which layers of a small model on the CPU are taken for alike once ``change`` has been at it, and the model and its notes."""
    from types import SimpleNamespace as Some
    from alofa_amd.config import config_from_dict
    from alofa_amd.engine.tapes import LayerTapes
    from alofa_amd.model import Model
    from alofa_amd.parts.base import Runtime
    config = config_from_dict({**MODEL, "num_hidden_layers": layers, "hidden_size": 64, "num_attention_heads": 2, "num_key_value_heads": 1, "intermediate_size": 64, "vocab_size": 20})
    w = {"model.embed_tokens.weight": torch.zeros(20, 64), "model.norm.weight": torch.ones(64)}
    for i in range(layers):
        pre = f"model.layers.{i}."
        for n, rows, cols in (("self_attn.q_proj", 64, 64), ("self_attn.k_proj", 32, 64), ("self_attn.v_proj", 32, 64), ("self_attn.o_proj", 64, 64), ("mlp.gate_proj", 64, 64), ("mlp.up_proj", 64, 64), ("mlp.down_proj", 64, 64)):
            w[pre + n + ".weight"] = torch.zeros(rows, cols, dtype=torch.bfloat16)
            if n[-6] in "qkv" and n.startswith("self"):
                w[pre + n + ".bias"] = torch.zeros(rows)
        for n in ("input_layernorm", "post_attention_layernorm"):
            w[pre + n + ".weight"] = torch.ones(64)
    model = Model(config.spec(), w, Runtime(torch.device("cpu"), torch.bfloat16))
    cache = Some(tensors={(i, 0): {"k": torch.zeros(8), "v": torch.zeros(8)} for i in range(layers)}, group_of_entry={(i, 0): 0 for i in range(layers)})
    change(model)
    made = LayerTapes.of(model, cache)
    return {} if made is None else made.source, model, made, cache


def test_which_layers_are_alike():
    assert alike()[0] == {2: 1, 3: 1, 4: 1}      # (the first has the embedding in front of it, the last no layer behind)

    def other_numbers(model):
        for i, b in enumerate(model.blocks):
            b.mixer.numbers = np.arange(5000) * (2 if i == 3 else 1)      # (alike at either end, as an array is written out)
            b.mixer.numbers[[*range(10), *range(-10, 0)]] = 0
    assert alike(other_numbers)[0] == {2: 1} or alike(other_numbers)[0] == {}
    assert 3 not in alike(other_numbers)[0]

    def named(model):
        for i, b in enumerate(model.blocks):
            b.feed_forward.more = {"w": torch.zeros(4, 4) if i != 3 else torch.zeros(4, 5), "rest": [1.0, None]}
    assert 3 not in alike(named)[0] and alike(lambda m: [setattr(b.feed_forward, "more", {"w": torch.zeros(4, 4)}) for b in m.blocks])[0] == {2: 1, 3: 1, 4: 1}
    shared, own = object(), [object() for _ in range(6)]
    assert alike(lambda m: [setattr(b.mixer, "x", shared) for b in m.blocks])[0] == {2: 1, 3: 1, 4: 1}
    assert alike(lambda m: [setattr(b.mixer, "x", x) for b, x in zip(m.blocks, own)])[0] == {}


def test_a_class_says_for_itself_that_it_may_be_run_so():
    from alofa_amd.parts.feed_forward import SwiGLU

    class Sum(SwiGLU):
        def forward(self, ctx, x, residual, **how):
            residual += x
    assert alike(lambda m: [setattr(b.feed_forward, "__class__", Sum) for b in m.blocks])[0] == {}


def test_matrices_that_are_replaced():
    """Behind the step function: its steps go through the parts. Another step function of the model has the new one."""
    from alofa_amd.engine.tapes import LayerTapes
    source, model, made, cache = alike()
    assert made.stand()
    model.blocks[3].feed_forward.w_down = torch.ones(64, 64, dtype=torch.bfloat16)
    assert not made.stand()
    again = LayerTapes.of(model, cache)
    assert again.source == source and again.stand() and model.blocks[3].feed_forward.w_down.data_ptr() in again.addresses(3) and model.blocks[3].feed_forward.w_down.data_ptr() not in made.addresses(3)
    model.blocks[2].norms[1] = model.blocks[1].norms[1]
    assert not again.stand()
    _, model, made, cache = alike()
    model.blocks[4].mixer.window = 40
    assert LayerTapes.of(model, cache).source == {2: 1}      # (three has another layer behind it then)


def test_what_is_asked_of_the_library_is_no_launch():
    """Launches are noted by ``_call``: what ops asks by ``_answer`` takes no stream."""
    import re
    from conftest import ROOT
    ops = (ROOT / "alofa_amd" / "ops.py").read_text()
    code = "\n".join(f.read_text() for f in sorted((ROOT / "alofa_amd" / "csrc").glob("*.hip")))
    asked = set(re.findall(r'_answer\("(\w+)"', ops)) | set(re.findall(r"load\(\)\.(alofa_\w+)\(", ops))
    assert len(asked) >= 6
    for name in asked:
        found = re.search(r'extern "C" [\w* ]+?\b' + name + r"\(([^)]*)\)", code)
        assert found and "hipStream_t" not in found.group(1), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("config", [MODEL, WINDOWS], ids=["alike", "two kinds of layers"])
def test_steps_are_the_same_bits_with_and_without_tapes(tmp_path, config, dtype, monkeypatch):
    from alofa_amd.engine import tapes
    from alofa_amd.replay import Replayer
    from alofa_amd.weights import write_random_model
    write_random_model(config, tmp_path, seed=5)
    rng = np.random.default_rng(3)
    ids = lambda n: [int(x) for x in rng.integers(0, 500, n)]      # noqa: E731
    # short prompts, a longer one, portions beside tokens that decode, and decode steps (which run once launch by launch and are then captured)
    steps = [[("a", ids(5)), ("b", ids(33))], [("c", ids(150))], [("a", ids(1)), ("b", ids(7)), ("c", ids(90))], [("a", ids(1)), ("b", ids(1)), ("c", ids(1))]] + [[("a", ids(1)), ("b", ids(1)), ("c", ids(1))]] * 2
    got = {}
    for on in (False, True):
        monkeypatch.setattr(tapes, "SWITCHED_ON", on)
        r = Replayer(str(tmp_path), dtype, 512)
        r.fn.resident = None
        assert (r.fn.tapes is not None) == on
        if on:
            assert r.fn.tapes.source == ({i: 1 for i in range(2, 6)} if config is MODEL else {4: 3, 5: 3})
        got[on] = [r.step({"step": k, "entries": [{"id": n, "tokens": t, "want": [len(t) - 1]} for n, t in s], "end": []}) for k, s in enumerate(steps)]
    for a, b in zip(got[False], got[True]):
        assert a.size and np.array_equal(a, b)
