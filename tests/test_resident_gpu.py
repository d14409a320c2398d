"""Decode steps whose layers run in one launch (csrc/decode_resident.hip), beside the kernels that run them one after the other and the 32-bit path."""
import numpy as np
import pytest
import torch

from alofa_amd.engine.step import StepEntry

pytestmark = pytest.mark.gpu

VOCAB, LAYERS = 512, 3


def model(width, heads, kv_heads, ff, dtype, layers=LAYERS, window=None, device="cuda:0", positions=4096):
    from alofa_amd.config import config_from_dict
    from alofa_amd.model import Model, runtime
    config = config_from_dict({"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "num_hidden_layers": layers, "hidden_size": width, "num_attention_heads": heads,
                               "num_key_value_heads": kv_heads, "head_dim": width // heads, "intermediate_size": ff, "vocab_size": VOCAB, "rope_theta": 10000.0, "rms_norm_eps": 1e-6,
                               "tie_word_embeddings": True, "use_sliding_window": window is not None, "max_position_embeddings": positions,
                               **({"sliding_window": window, "max_window_layers": 0} if window else {})})
    gen = torch.Generator(device="cuda").manual_seed(7)

    def draw(*shape, scale=1.0, shift=0.0):
        return (torch.randn(shape, generator=gen, device="cuda") * scale + shift).to(torch.bfloat16)
    d = width // heads
    w = {"model.embed_tokens.weight": draw(VOCAB, width), "model.norm.weight": draw(width, scale=0.1, shift=1.0)}
    for i in range(layers):
        pre = f"model.layers.{i}."
        for n, rows, cols in (("self_attn.q_proj", heads * d, width), ("self_attn.k_proj", kv_heads * d, width), ("self_attn.v_proj", kv_heads * d, width),
                              ("self_attn.o_proj", width, heads * d), ("mlp.gate_proj", ff, width), ("mlp.up_proj", ff, width), ("mlp.down_proj", width, ff)):
            w[pre + n + ".weight"] = draw(rows, cols, scale=cols ** -0.5)
            if n[-6] in "qkv" and n.startswith("self"):
                w[pre + n + ".bias"] = draw(rows, scale=0.5)
        for n in ("input_layernorm", "post_attention_layernorm"):
            w[pre + n + ".weight"] = draw(width, scale=0.1, shift=1.0)
    return config, Model(config.spec(), w, runtime(dtype, device))


def engine(m, rows, context, dtype, page=16):
    from alofa_amd import Engine
    return Engine(None, dtype=dtype, max_tokens=context + 8, max_batch=rows, kv_blocks=rows * ((context + 8) // page + 2), block_size=page, token_budget=4096, watermark_permille=1000, model=m)


def stand(eng, lengths, seed):
    """Requests 0.. with lengths[i] tokens in the cache."""
    rng = np.random.default_rng(seed)
    for i, n in enumerate(lengths):
        eng.cache.admit(i)
        for at in range(0, n, 4096):      # (no more than a step's tokens at once)
            eng.step_fn.run([StepEntry(i, rng.integers(0, VOCAB, min(n - at, 4096)).tolist())])


def decode(eng, tokens):
    return [eng.step_fn.run([StepEntry(i, [int(t)], [0]) for i, t in enumerate(row)]).double().cpu() for row in tokens]


# widths: the least, ones whose columns do not divide by the blocks, the most; keys at the edges of tiles, pages, parts and a wave's first step
SHAPES = [(256, 4, 1, 512), (320, 5, 5, 768), (896, 14, 2, 4864), (1024, 16, 2, 6144)]
CONTEXTS = [0, 1, 15, 16, 17, 31, 255, 256, 300, 511, 600, 1023, 7, 48, 130, 2100]


@pytest.mark.parametrize("page", [16, 64])
@pytest.mark.parametrize("rows", [1, 2, 3, 5, 8, 9, 16])
@pytest.mark.parametrize("shape", SHAPES)
def test_one_launch_is_as_near_the_32_bit_path_as_the_kernels_it_replaces(shape, rows, page):
    lengths = (CONTEXTS * 2)[rows:2 * rows] if rows < 16 else CONTEXTS
    tokens = np.random.default_rng(rows).integers(0, VOCAB, (3, rows))
    got = {}
    for how in ("float32", "one by one", "one launch", "one launch, captured"):
        dtype = "float32" if how == "float32" else "bfloat16"
        m = model(*shape, dtype)
        eng = engine(m, rows, max(lengths) + 4, dtype, page)
        fn = eng.step_fn
        assert (fn.resident is None) == (how == "float32")
        if how == "one by one":
            fn.resident = None
        fn.use_graphs = how.endswith("captured")
        stand(eng, lengths, 1)
        got[how] = decode(eng, tokens)
        if how.endswith("captured"):
            assert fn.graph_replays > 0
    for step in range(len(tokens)):
        exact = got["float32"][step]
        off = {how: ((x[step] - exact).norm() / exact.norm()).item() for how, x in got.items()}
        # both round the same values to bfloat16 and add in float32 in orders of their own: roundings that fall the other way are as many on either side, and
        # over at least 512 logits the two distances are alike within a third (the spread of a norm of that many independent errors, with those of a layer's rows shared)
        assert off["one launch"] <= 1.34 * off["one by one"] + 1e-4, (step, off)
        # the same kernel on the same cache, whether captured or not
        a, b = got["one launch"][step], got["one launch, captured"][step]
        assert torch.equal(a, b), (step, (a != b).sum(1).tolist(), (a - b).abs().amax(1).tolist(), lengths)


@pytest.mark.parametrize("name", ["k", "v"])
def test_a_cached_key_or_value_that_is_no_number_reaches_the_logits(name):
    """NaN in one request's cache, in its first tile of keys, one in the middle and its last: that row is NaN, the others keep their bits."""
    lengths, page = [300, 40, 600], 16
    tokens = [[5, 6, 7]]
    m = model(896, 14, 2, 4864, "bfloat16")
    eng = engine(m, 3, 700, "bfloat16", page)
    stand(eng, lengths, 9)
    clean = decode(eng, tokens)[0]
    for at in (3, 299, 590):
        eng = engine(m, 3, 700, "bfloat16", page)
        stand(eng, lengths, 9)
        block = eng.cache.table(2, 0)[at // page]
        t = eng.cache.tensors[(1, 0)][name]
        (t[block, 1, at % page] if name == "k" else t[block, 1, :, at % page]).fill_(float("nan"))
        got = decode(eng, tokens)[0]
        assert torch.isnan(got[2]).all() and torch.equal(got[:2], clean[:2]), at


def test_steps_in_turn_do_not_disturb_one_another():
    """Two engines with areas of their own, of different rows, and steps that are no decode steps in between."""
    tokens = np.random.default_rng(3).integers(0, VOCAB, (12, 8))
    m = model(896, 14, 2, 4864, "bfloat16")
    alone = {}
    for rows in (2, 8):
        eng = engine(m, rows, 100, "bfloat16")
        stand(eng, [33 + i for i in range(rows)], 5)
        alone[rows] = decode(eng, tokens[:, :rows])
    both = {rows: engine(m, rows, 100, "bfloat16") for rows in (2, 8)}
    assert both[2].step_fn.resident.area != both[8].step_fn.resident.area
    for rows, eng in both.items():
        stand(eng, [33 + i for i in range(rows)], 5)
    for k, row in enumerate(tokens):
        for rows, eng in both.items():
            assert torch.equal(decode(eng, row[None, :rows])[0], alone[rows][k]), (k, rows)


def test_threads_with_streams_of_their_own_take_turns():
    import threading
    tokens = np.random.default_rng(4).integers(0, VOCAB, (40, 8))
    m = model(896, 14, 2, 4864, "bfloat16")
    sizes = (1, 3, 8, 2)
    want = []
    for rows in sizes:
        eng = engine(m, rows, 100, "bfloat16")
        stand(eng, [20 + i for i in range(rows)], 6)
        want.append(torch.stack(decode(eng, tokens[:, :rows])))
    engines = [engine(m, rows, 100, "bfloat16") for rows in sizes]
    for rows, eng in zip(sizes, engines):
        stand(eng, [20 + i for i in range(rows)], 6)
        decode(eng, tokens[:1, :rows])      # (captured here: a capture forbids what other threads may be doing)
    torch.cuda.synchronize()
    got, start = {}, threading.Barrier(len(sizes))

    def run(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait()
                got[k] = torch.stack(decode(engines[k], tokens[1:, :sizes[k]]))
        except BaseException as e:
            got[k] = e
    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(sizes))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for k in range(len(sizes)):
        assert isinstance(got[k], torch.Tensor), got[k]
        assert torch.equal(got[k], want[k][1:]), k


def test_what_it_does_not_take_runs_kernel_by_kernel():
    assert engine(model(896, 14, 2, 4864, "bfloat16"), 2, 64, "bfloat16").step_fn.resident is not None
    assert engine(model(896, 14, 2, 4864, "float32"), 2, 64, "float32").step_fn.resident is None
    assert engine(model(896, 14, 2, 4864, "bfloat16", window=32), 2, 64, "bfloat16").step_fn.resident is None
    assert engine(model(896, 14, 2, 4864, "bfloat16"), 2, 64, "bfloat16", page=8).step_fn.resident is None      # (pages of fewer than 16 tokens)
    assert engine(model(512, 4, 1, 1024, "bfloat16"), 2, 64, "bfloat16").step_fn.resident is None               # heads of 128
    assert engine(model(192, 3, 1, 512, "bfloat16"), 2, 64, "bfloat16").step_fn.resident is None                # fewer columns than blocks
    eng = engine(model(896, 14, 2, 4864, "bfloat16"), 24, 64, "bfloat16")
    stand(eng, [5] * 17, 2)
    before = eng.step_fn.resident.failed.item()
    assert all(torch.isfinite(x).all() for x in decode(eng, np.ones((2, 17), dtype=int)))      # (17 rows)
    assert before == 0 and eng.step_fn.resident.failed.item() == 0


def test_areas_are_used_again():
    import gc
    from alofa_amd.engine.resident import _areas
    m = model(256, 4, 1, 512, "bfloat16", layers=1)
    eng = engine(m, 1, 32, "bfloat16")
    stand(eng, [3], 1)
    area, want = eng.step_fn.resident.area, decode(eng, [[1], [2]])
    del eng
    gc.collect()
    idle = [a for areas in _areas._idle.values() for a in areas]
    assert area in idle
    eng = engine(m, 1, 32, "bfloat16")
    assert eng.step_fn.resident.area in idle
    stand(eng, [3], 1)
    assert all(torch.equal(a, b) for a, b in zip(decode(eng, [[1], [2]]), want))


def write(address, words):
    """64-bit words into device memory that no tensor stands for."""
    import ctypes
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    block = (ctypes.c_uint64 * len(words))(*words)
    assert hip.hipMemcpy(ctypes.c_void_p(address), block, ctypes.c_size_t(8 * len(words)), 1) == 0      # (1: host to device)


def test_the_area_of_a_step_function_that_failed_serves_the_next_one():
    """What such a launch leaves behind, written by the host: the stop word, a counter that has gone on, values that bear the numbers of steps to come."""
    import gc
    from alofa_amd.engine.resident import _areas
    m = model(256, 4, 1, 512, "bfloat16", layers=2)
    tokens = [[1], [2], [3]]

    def run():
        eng = engine(m, 1, 32, "bfloat16")
        stand(eng, [3], 1)
        return eng, decode(eng, tokens)
    gc.collect()
    _areas._idle.clear()      # (those of other tests stay out of it)
    eng, want = run()
    area, address = eng.step_fn.resident.area, eng.step_fn.resident.area.address
    torch.cuda.synchronize()
    write(address, [6, 1] + [0] * 30 + [(7 + i % 5) << 32 | 0x3f800000 for i in range(400000)])      # (all of the places, with numbers that come next)
    area.failed[0] = 1
    del eng, area
    gc.collect()
    eng, got = run()
    assert eng.step_fn.resident.area.address == address
    assert all(torch.equal(a, b) for a, b in zip(got, want)), [torch.isnan(x).any().item() for x in got]
    assert eng.step_fn.resident.failed.item() == 0


def test_a_wait_given_up_is_an_error_of_the_next_step():
    """The word that the kernel sets, set by the host."""
    from alofa_amd.errors import AlofaError
    eng = engine(model(256, 4, 1, 512, "bfloat16", layers=1), 1, 32, "bfloat16")
    stand(eng, [3], 1)
    assert torch.isfinite(decode(eng, [[1]])[0]).all()
    eng.step_fn.resident.failed[0] = 1
    with pytest.raises(AlofaError):
        decode(eng, [[1]])


@pytest.mark.parametrize("how", [{}, {"temperature": 0.8}, {"temperature": 0.8, "top_k": 5}])
@pytest.mark.parametrize("last", [True, False])
def test_tokens_of_a_step_that_gave_up_do_not_come_out(how, last):
    """The word that the kernel sets, set by the host while the step is on its way: the last step of a run, or one before it."""
    from alofa_amd.errors import LostResults
    eng = engine(model(256, 4, 1, 512, "bfloat16", layers=1), 2, 32, "bfloat16")
    steps, run = [], eng.step_fn.run

    def failing(entries, greedy=False):
        out = run(entries, greedy)
        steps.append(len(entries))
        if len(steps) == (4 if last else 2):
            eng.step_fn.resident.failed[0] = 1
        return out
    eng.step_fn.run = failing
    with pytest.raises(LostResults):
        eng.generate([[5, 6, 7], [8, 9]], max_new=4, **how)
    assert len(steps) <= (4 if last else 3)
    for r in eng.core.requests:
        with pytest.raises(LostResults):
            eng.core.output(r)


@pytest.mark.parametrize("captured", [True, False])
def test_behind_a_step_that_gave_up_all_steps_run_kernel_by_kernel(captured):
    from alofa_amd.errors import LostResults
    m = model(896, 14, 2, 4864, "bfloat16")
    tokens = np.random.default_rng(8).integers(0, VOCAB, (4, 3))
    engines = {}
    for how in ("one by one", "gave up"):
        eng = engines[how] = engine(m, 3, 100, "bfloat16")
        eng.step_fn.use_graphs = captured
        if how == "one by one":
            eng.step_fn.resident = None
        else:
            eng.cache.admit("before")
            eng.step_fn.run([StepEntry("before", [5], [0])])
            eng.step_fn.run([StepEntry("before", [6], [0])])
            eng.step_fn.resident.failed[0] = 1
            with pytest.raises(LostResults):
                eng.step_fn.run([StepEntry("before", [7], [0])])
            assert eng.step_fn.resident is None
            eng.cache.free("before")
        stand(eng, [33, 5, 70], 2)
    replayed = engines["gave up"].step_fn.graph_replays
    want, got = (decode(engines[how], tokens) for how in ("one by one", "gave up"))
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    assert (engines["gave up"].step_fn.graph_replays > replayed) == captured


def test_without_a_seat_or_switched_off_steps_run_kernel_by_kernel(monkeypatch):
    from alofa_amd.engine import resident
    m = model(256, 4, 1, 512, "bfloat16", layers=1)
    monkeypatch.setattr(resident._seats, "take", lambda gpu: False)
    assert engine(m, 1, 32, "bfloat16").step_fn.resident is None
    monkeypatch.undo()
    monkeypatch.setenv("ALOFA_ONE_LAUNCH", "0")
    assert engine(m, 1, 32, "bfloat16").step_fn.resident is None
    monkeypatch.undo()
    assert engine(m, 1, 32, "bfloat16").step_fn.resident is not None


def test_prompts_in_one_thread_and_decode_steps_in_others():
    """Each with a stream of its own, the decode steps laid out and launched one by one (sizes whose kernels hand nothing over in the library's workspace, which is for one stream at a time)."""
    import threading
    m = model(256, 4, 1, 512, "bfloat16", layers=2)
    rng = np.random.default_rng(12)
    tokens, prompts = rng.integers(0, VOCAB, (30, 3)), rng.integers(0, VOCAB, (30, 9)).tolist()

    def prompt_steps(eng):
        out = []
        for p in prompts:
            eng.cache.admit(0)
            out.append(eng.step_fn.run([StepEntry(0, p, [8])]).double().cpu())
            eng.cache.free(0)
        return torch.stack(out)

    def engines():
        made = {n: engine(m, 3, 64, "bfloat16") for n in ("prompts", 2, 3)}
        for n, eng in made.items():
            eng.step_fn.use_graphs = False
            if n != "prompts":
                stand(eng, [11 + i for i in range(n)], 7)
        torch.cuda.synchronize()
        return made

    def work(n, eng):
        return prompt_steps(eng) if n == "prompts" else torch.stack(decode(eng, tokens[:, :n]))
    want = {n: work(n, eng) for n, eng in engines().items()}
    got, start = {}, threading.Barrier(3)

    def run(n, eng):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait()
                got[n] = work(n, eng)
        except BaseException as e:
            got[n] = e
    threads = [threading.Thread(target=run, args=x) for x in engines().items()]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for n in want:
        assert isinstance(got[n], torch.Tensor), got[n]
        assert torch.equal(got[n], want[n]), n


@pytest.mark.parametrize("shape,rows", [((256, 4, 1, 512), 1), ((320, 5, 5, 768), 5), ((896, 14, 2, 4864), 2), ((896, 14, 2, 4864), 9), ((1024, 16, 2, 6144), 16)])
def test_no_number_comes_from_a_wait_that_was_given_up(shape, rows):
    """Waits given up after 1 to 40 asks, of which an ordinary one takes a few: each row is the right one or has NaN in it, and if one is not the right one, the
    word says that a wait was given up. Every launch ends."""
    from alofa_amd import ops
    m = model(*shape, "bfloat16")
    lengths = (CONTEXTS * 2)[3:3 + rows]
    eng = engine(m, rows, max(lengths) + 4, "bfloat16")
    stand(eng, lengths, 4)
    fn, res = eng.step_fn, eng.step_fn.resident
    ctx, ids, _ = fn.begin([StepEntry(i, [7 + i], [0]) for i in range(rows)])
    start = m[1].embedding.forward(ctx, ids).clone()
    cos, sin = res.position.table(ctx.n_positions)

    def run(limit):
        ops.clear_resident_area(res.area.address)
        res.failed.zero_()
        hidden = start.clone()
        ops.decode_resident(hidden, res.layers, ctx.positions, ctx._tables[res.group], ctx._slots[res.group], cos, sin, res.area.address, res.failed, res.intermediate,
                            res.heads, res.kv_heads, res.d, res.page, res.biased, res.scale, res.eps, limit=limit)
        torch.cuda.synchronize()
        return hidden, bool(res.failed.item())
    want, failed = run(0)
    assert torch.isfinite(want).all() and not failed
    given_up = 0
    for limit in [*range(1, 41), 1, 1, 2, 2, 3, 3]:
        got, failed = run(limit)
        given_up += failed
        right = (got == want).all(1)
        assert (right | torch.isnan(got).any(1)).all(), (limit, failed)
        assert failed or right.all(), limit
    assert given_up > 0      # (a first ask that finds every value there, in every block and phase, is not to be had)
    ops.clear_resident_area(res.area.address)
    res.failed.zero_()
    assert torch.equal(run(0)[0], want)


def ends(work):
    """``work`` in a thread of its own, whose end is waited for, but not for ever; what it returned."""
    import threading
    got = []

    def run():
        try:
            got.append(work())
        except BaseException as e:
            got.append(e)
    th = threading.Thread(target=run, daemon=True)
    th.start()
    th.join(30)
    assert got, "still waiting"
    assert not isinstance(got[0], BaseException), got[0]
    return got[0]


def test_a_step_within_a_step_that_is_watched():
    m = model(256, 4, 1, 512, "bfloat16", layers=2)
    outer, inner = (engine(m, 2, 64, "bfloat16") for _ in range(2))
    stand(outer, [5, 9], 1), stand(inner, [12], 1)
    seen = []
    outer.step_fn.watch = lambda i, hidden: seen.append(decode(inner, [[i]])[0])
    got = ends(lambda: decode(outer, [[1, 2]]))
    assert len(seen) == 2 and all(torch.isfinite(x).all() for x in [*seen, *got])


def test_a_step_that_is_being_laid_out_keeps_no_other_waiting():
    import threading
    m = model(256, 4, 1, 512, "bfloat16", layers=2)
    slow, other = (engine(m, 1, 64, "bfloat16") for _ in range(2))
    stand(slow, [5], 1), stand(other, [9], 1)
    decode(other, [[3]])      # (captured)
    inside, go_on, plan = threading.Event(), threading.Event(), slow.step_fn.plan

    def plan_slowly(entries):
        inside.set()
        go_on.wait(60)
        return plan(entries)
    slow.step_fn.plan = plan_slowly
    th = threading.Thread(target=lambda: decode(slow, [[1]]), daemon=True)
    th.start()
    assert inside.wait(30)
    try:
        ends(lambda: decode(other, [[4], [5]]))
    finally:
        go_on.set()
        th.join(30)
    assert not th.is_alive()


@pytest.mark.parametrize("how", ["stored in 32 bits", "one matrix in 32 bits", "off its place"])
def test_matrices_that_the_launch_cannot_read_run_kernel_by_kernel(how, monkeypatch):
    """Matrices keep the type they were stored in and the place they were given: the results are those of the kernels one by one."""
    config, first = model(256, 4, 1, 512, "bfloat16", layers=2)
    from alofa_amd.model import Model, runtime

    def shifted(t):
        room = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        return room[1:].view(t.shape).copy_(t)
    weights = {}
    for i, b in enumerate(first.blocks):
        pre, q, kv = f"model.layers.{i}.", 4 * 64, 64
        for n, t in zip("qkv", b.mixer.w_qkv.split([q, kv, kv])):
            weights[pre + f"self_attn.{n}_proj.weight"] = t
        for n, t in zip("qkv", b.mixer.b_qkv.split([q, kv, kv])):
            weights[pre + f"self_attn.{n}_proj.bias"] = t
        weights.update({pre + "self_attn.o_proj.weight": b.mixer.w_o, pre + "mlp.gate_proj.weight": b.feed_forward.w_gate, pre + "mlp.up_proj.weight": b.feed_forward.w_up,
                        pre + "mlp.down_proj.weight": b.feed_forward.w_down, pre + "input_layernorm.weight": b.norms[0].weight, pre + "post_attention_layernorm.weight": b.norms[1].weight})
    weights.update({"model.embed_tokens.weight": first.embedding.table, "model.norm.weight": first.final_norm.weight})
    for n, t in weights.items():
        if t.dim() == 2 and (how == "stored in 32 bits" or (how == "one matrix in 32 bits" and n == "model.layers.1.mlp.down_proj.weight")):
            weights[n] = t.float()
        elif how == "off its place" and n == "model.layers.1.self_attn.o_proj.weight":
            weights[n] = shifted(t)
    m = config, Model(config.spec(), weights, runtime("bfloat16"))
    got = {}
    for switch in ("1", "0"):
        monkeypatch.setenv("ALOFA_ONE_LAUNCH", switch)
        eng = engine(m, 2, 64, "bfloat16")
        assert eng.step_fn.resident is None
        stand(eng, [5, 20], 3)
        got[switch] = decode(eng, [[1, 2], [3, 4]])
    assert all(torch.equal(a, b) and torch.isfinite(a).all() for a, b in zip(got["1"], got["0"]))


def test_without_memory_for_an_area_steps_run_kernel_by_kernel(monkeypatch):
    from alofa_amd import ops
    from alofa_amd.engine import resident
    from alofa_amd.errors import AlofaError

    def none():
        raise AlofaError("capacity", "no memory for an area")
    m = model(256, 4, 1, 512, "bfloat16", layers=1)
    monkeypatch.setattr(resident, "_areas", resident._Areas())
    monkeypatch.setattr(ops, "resident_area", none)
    eng = engine(m, 1, 32, "bfloat16")
    assert eng.step_fn.resident is None
    stand(eng, [3], 1)
    assert torch.isfinite(decode(eng, [[1]])[0]).all()


def test_a_gpu_named_without_its_number_is_the_same_gpu():
    config, first = model(256, 4, 1, 512, "bfloat16", layers=1)
    turns = [engine(m, 1, 32, "bfloat16").step_fn.resident.turn for m in ((config, first), model(256, 4, 1, 512, "bfloat16", layers=1, device="cuda"))]
    assert turns[0] is turns[1]


def test_a_step_that_grows_past_the_keys_it_is_for(monkeypatch):
    """In the middle of a captured length (one graph for either way), laid out eagerly and captured: the same bits."""
    from alofa_amd.engine.resident import ResidentLayers
    monkeypatch.setattr(ResidentLayers, "MOST_KEYS", ((4, 40), (16, 1000)))
    m = model(256, 4, 1, 512, "bfloat16", layers=2)
    got = {}
    for captured in (True, False):
        eng = engine(m, 2, 100, "bfloat16")
        eng.step_fn.use_graphs = captured
        stand(eng, [37, 20], 5)
        got[captured] = decode(eng, np.arange(14).reshape(7, 2))
        if captured:
            assert {key[3] for key in eng.step_fn._graphs} == {True, False} and eng.step_fn.graph_replays == 5
    assert all(torch.equal(a, b) and torch.isfinite(a).all() for a, b in zip(got[True], got[False]))


def test_generate_again_behind_a_step_that_gave_up():
    """More prompts than the pages hold at once, so that some have not begun when it happens: the next call's results are its own."""
    from alofa_amd import Engine
    from alofa_amd.errors import LostResults
    m = model(256, 4, 1, 512, "bfloat16", layers=2)
    prompts = np.random.default_rng(6).integers(0, VOCAB, (6, 40)).tolist()
    engines = [Engine(None, dtype="bfloat16", max_tokens=64, max_batch=6, kv_blocks=9, block_size=16, token_budget=64, watermark_permille=1000, model=m) for _ in range(2)]
    engines[0].step_fn.resident = None
    want = engines[0].generate(prompts[3:], max_new=6)
    eng, run = engines[1], engines[1].step_fn.run
    steps = []

    def failing(entries, greedy=False):
        out = run(entries, greedy)
        steps.append(entries)
        if len(steps) == 6:
            eng.step_fn.resident.failed[0] = 1
        return out
    eng.step_fn.run = failing
    with pytest.raises(LostResults):
        eng.generate(prompts, max_new=6)
    assert eng.generate(prompts[3:], max_new=6) == want
    assert not eng.core.has_work() and not eng.core.cache.requests


# more than sixteen rows (csrc/decode_groups.hip): the least and most of two and of four groups, groups of unlike sizes; widths: the least, one whose pairs of columns do not divide by the
# blocks and that stays at 32 rows for its key heads, one between, the 0.5B sizes, the most
GROUP_SHAPES = [(256, 4, 1, 512), (320, 5, 5, 768), (576, 9, 3, 1536), (896, 14, 2, 4864), (1024, 16, 4, 4096)]


@pytest.mark.parametrize("page", [16, 64])
@pytest.mark.parametrize("rows", [17, 31, 32, 33, 50, 64])
@pytest.mark.parametrize("shape", GROUP_SHAPES)
def test_groups_are_as_near_the_32_bit_path_as_the_kernels_they_replace(shape, rows, page, monkeypatch):
    lengths = (CONTEXTS * 4)[rows % 5:][:rows] + [33] * (rows - len((CONTEXTS * 4)[rows % 5:][:rows]))
    groups_beside_the_32_bit_path(shape, lengths, page, monkeypatch)


@pytest.mark.parametrize("rows", [17, 33])
@pytest.mark.parametrize("shape", [(256, 4, 1, 512), (512, 8, 2, 1024)])
def test_a_row_of_more_keys_than_its_parts_are_for_beside_short_ones(shape, rows, monkeypatch):
    """The most parts that a row and key head has, sixteen, each of more tiles of keys than the group's other blocks, and all rounds of the launch's sums over parts."""
    groups_beside_the_32_bit_path(shape, [40 + 13 * i for i in range(rows // 2)] + [6100] + [15 + i for i in range(rows - rows // 2 - 1)], 16, monkeypatch)


def counted(monkeypatch) -> list:
    """The rows of every launch from here on."""
    from alofa_amd import ops
    launches, one_launch = [], ops.decode_resident
    monkeypatch.setattr(ops, "decode_resident", lambda hidden, *a, **how: (launches.append(hidden.shape[0]), one_launch(hidden, *a, **how))[1])
    return launches


def groups_beside_the_32_bit_path(shape, lengths, page, monkeypatch):
    rows, launches = len(lengths), counted(monkeypatch)
    tokens = np.random.default_rng(rows).integers(0, VOCAB, (2, rows))
    got = {}
    for how in ("float32", "one by one", "one launch", "one launch, captured"):
        dtype = "float32" if how == "float32" else "bfloat16"
        eng = engine(model(*shape, dtype, layers=2, positions=8192), rows, max(lengths) + 4, dtype, page)
        fn = eng.step_fn
        if how.startswith("one launch"):
            assert fn.resident.most_rows == (32 if shape[2] > 4 else 64)
        if how == "one by one":
            fn.resident = None
        fn.use_graphs = how.endswith("captured")
        stand(eng, lengths, 1)
        launches.clear()
        got[how] = decode(eng, tokens)
        # (captured: a step that replays no graph launches once for its results and once for the graph)
        steps = 2 * (len(tokens) - fn.graph_replays) if how.endswith("captured") else len(tokens)
        # (five key heads: 32 rows at most, and kernel by kernel beyond)
        assert launches == ([rows] * steps if how.startswith("one launch") and rows <= fn.resident.most_rows else []), (how, launches)
    for step in range(len(tokens)):
        exact = got["float32"][step]
        # (per row: a row that took another's place would hide among so many; the spread of the norm of 512 logits' roundings, as above, is less than a third of it)
        off = {how: ((x[step] - exact).norm(dim=1) / exact.norm(dim=1)) for how, x in got.items()}
        assert (off["one launch"] <= 1.6 * off["one by one"].mean() + 1e-4).all(), (step, off["one launch"].max(), off["one by one"].max())
        assert off["one launch"].norm() <= 1.34 * off["one by one"].norm() + 1e-4
        assert torch.equal(got["one launch"][step], got["one launch, captured"][step]), step


@pytest.mark.parametrize("shape,rows", [((256, 4, 1, 512), 17), ((896, 14, 2, 4864), 32), ((896, 14, 2, 4864), 64)])
def test_no_number_of_a_group_comes_from_a_wait_that_was_given_up(shape, rows):
    """As above, in groups, each of which may give up by itself."""
    from alofa_amd import ops
    m = model(*shape, "bfloat16", layers=2)
    lengths = [20 + 7 * i for i in range(rows)]
    eng = engine(m, rows, max(lengths) + 4, "bfloat16")
    stand(eng, lengths, 4)
    fn, res = eng.step_fn, eng.step_fn.resident
    ctx, ids, _ = fn.begin([StepEntry(i, [7 + i], [0]) for i in range(rows)])
    start = m[1].embedding.forward(ctx, ids).clone()
    cos, sin = res.position.table(ctx.n_positions)

    def run(limit):
        ops.clear_resident_area(res.area.address)
        res.failed.zero_()
        hidden = start.clone()
        ops.decode_resident(hidden, res.layers, ctx.positions, ctx._tables[res.group], ctx._slots[res.group], cos, sin, res.area.address, res.failed, res.intermediate,
                            res.heads, res.kv_heads, res.d, res.page, res.biased, res.scale, res.eps, limit=limit)
        torch.cuda.synchronize()
        return hidden, bool(res.failed.item())
    want, failed = run(0)
    assert torch.isfinite(want).all() and not failed
    given_up = 0
    for limit in [*range(1, 21), 1, 2, 3]:
        got, failed = run(limit)
        given_up += failed
        right = (got == want).all(1)
        assert (right | torch.isnan(got).any(1)).all(), (limit, failed)
        assert failed or right.all(), limit
    assert given_up > 0
    assert torch.equal(run(0)[0], want)


@pytest.mark.parametrize("name", ["k", "v"])
def test_a_cached_key_or_value_that_is_no_number_reaches_its_row_alone_in_a_group(name, monkeypatch):
    launches = counted(monkeypatch)
    lengths, page = [300, 40, 600] + [25 + i for i in range(17)], 16
    tokens = [list(range(5, 25))]
    m = model(896, 14, 2, 4864, "bfloat16")
    eng = engine(m, 20, 700, "bfloat16", page)
    stand(eng, lengths, 9)
    clean = decode(eng, tokens)[0]
    others = [i for i in range(20) if i != 2]
    for at in (3, 299, 590):
        eng = engine(m, 20, 700, "bfloat16", page)
        stand(eng, lengths, 9)
        block = eng.cache.table(2, 0)[at // page]
        t = eng.cache.tensors[(1, 0)][name]
        (t[block, 1, at % page] if name == "k" else t[block, 1, :, at % page]).fill_(float("nan"))
        got = decode(eng, tokens)[0]
        assert torch.isnan(got[2]).all() and torch.equal(got[others], clean[others]), at
    assert set(launches) == {20}


def test_steps_of_few_and_of_many_rows_in_turn(monkeypatch):
    """One step function whose steps have 20, 3, 40 and 20 rows: the groups' counters go on apart from one another."""
    m = model(896, 14, 2, 4864, "bfloat16", layers=2)
    rng = np.random.default_rng(5)
    lengths = [30 + 3 * i for i in range(40)]
    counts = [20, 3, 40, 20, 3, 40, 40]
    tokens = [rng.integers(0, VOCAB, n).tolist() for n in counts]
    launches = counted(monkeypatch)

    def run(one_launch, graphs):
        eng = engine(m, 40, 300, "bfloat16")
        if not one_launch:
            eng.step_fn.resident = None
        eng.step_fn.use_graphs = graphs
        stand(eng, lengths, 3)
        return [eng.step_fn.run([StepEntry(i, [t], [0]) for i, t in enumerate(ts)]).double().cpu() for ts in tokens]
    want = run(False, False)
    assert not launches
    got = run(True, False)
    assert launches == counts
    captured = run(True, True)
    for a, b, c in zip(want, got, captured):
        assert ((a - b).norm() / a.norm()).item() < 0.02 and torch.equal(b, c)      # (two bfloat16 roundings of two layers: some 0.003 each)
