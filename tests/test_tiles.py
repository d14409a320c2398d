"""Matrices laid out in tiles for decode steps of more than sixteen rows in one launch."""
import numpy as np
import pytest
import torch


@pytest.mark.parametrize("n,k", [(16, 32), (48, 96), (80, 32)])
def test_where_a_value_lies_in_tiles(n, k):
    from alofa_amd import ops
    w = torch.arange(n * k).view(n, k)
    flat = ops.in_tiles(w).view(-1)
    for row in range(n):
        for col in range(k):
            lane = col % 32 // 8 * 16 + row % 16
            assert flat[((row // 16 * (k // 32) + col // 32) * 64 + lane) * 8 + col % 8] == w[row, col]
    again = torch.zeros_like(w)
    assert ops.in_tiles(w, again) is again and torch.equal(again.view(-1), flat)


def test_the_addresses_that_captured_steps_read_stay_where_they_are(monkeypatch):
    """A captured launch has the place of the layers' addresses in it: laying the tiles out moves nothing that it reads."""
    from types import SimpleNamespace as Some
    from alofa_amd import ops
    from alofa_amd.engine import resident
    from alofa_amd.model import Model
    monkeypatch.setattr(resident, "_areas", resident._Areas()), monkeypatch.setattr(resident, "_turns", {})
    monkeypatch.setattr(ops, "resident_rows", lambda *a: 64), monkeypatch.setattr(ops, "check_caches", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: Some(synchronize=lambda: None)), monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (1 << 40, 1 << 40)), monkeypatch.setattr(torch.cuda, "memory_reserved", lambda *a: 0), monkeypatch.setattr(torch.cuda, "memory_allocated", lambda *a: 0)
    mixer = Some(heads=4, kv_heads=1, d=64, scale=1.0, position=None, hidden=256, b_qkv=None)
    block = Some(mixer=mixer, feed_forward=Some(intermediate=512), norms=[Some(as_rmsnorm=lambda: (None, 1e-6))] * 2)
    tables = [[torch.zeros(1), None, torch.zeros(1), torch.zeros(512, 256), torch.zeros(512, 256), torch.zeros(256, 512), *(torch.zeros(1) for _ in range(4))] for _ in range(3)]
    model, cache = Model.__new__(Model), Some(block_size=16, group_of_entry={(0, 0): 0})
    model.tiles, model.written = None, 0
    layers = resident.ResidentLayers(model, [block] * 3, cache, torch.device("cpu"), tables, Some(failed=torch.zeros(1, dtype=torch.int32), address=0))
    held, at = layers._table, layers._table.data_ptr()
    before = held[0].clone()
    layers.ready(16)
    assert layers._tiles is None
    layers.ready(17)
    assert layers._tiles is not None
    assert layers._table is held and held.data_ptr() == at and torch.equal(held[0], before)
    assert [held[1, i, 3:6].tolist() for i in range(3)] == [[t.data_ptr() for t in layers._tiles.copies[3 * i:3 * i + 3]] for i in range(3)]
    assert torch.equal(held[1][:, [0, 1, 2, 6, 7, 8, 9]], before[:, [0, 1, 2, 6, 7, 8, 9]])


@pytest.mark.gpu
def test_a_captured_step_of_few_rows_behind_one_of_many():
    """Sixteen rows captured, seventeen, for which tiles are laid out, small tensors that take whatever memory was given back, and the captured steps of sixteen again: beside an engine whose tiles were
    there before its first step."""
    from test_resident_gpu import decode, engine, model, stand
    m, lengths = model(896, 14, 2, 1024, "bfloat16"), [11 * i for i in range(17)]
    tokens = np.random.default_rng(5).integers(0, 500, (9, 17)).tolist()
    steps = [tokens[i][:17 if i in (3, 7) else 16] for i in range(9)]
    got = []
    for first in (False, True):
        m[1].tiles = None
        e = engine(m, 17, 400, "bfloat16")
        if first:
            e.step_fn.resident.ready(17)
            assert m[1].tiles is not None
        stand(e, lengths, 1)
        out = decode(e, steps[:4])
        replays = e.step_fn.graph_replays
        held = [torch.full((n,), -1, dtype=torch.int64, device="cuda") for n in (30, 60, 60, 120, 250)]
        out += decode(e, steps[4:])
        assert e.step_fn.graph_replays == replays + 5 and all(bool((t == -1).all()) for t in held)
        got.append(out)
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [17, 40])
def test_matrices_written_in_place_are_laid_out_again(rows):
    from test_resident_gpu import decode, engine, model, stand
    shape, lengths = (256, 4, 1, 512), [9 * i for i in range(rows)]
    tokens = np.random.default_rng(3).integers(0, 500, (3, rows))
    m = model(*shape, "bfloat16")
    two = [engine(m, rows, max(lengths) + 12, "bfloat16") for _ in range(2)]
    for e in two:
        stand(e, lengths, 1)
    before = [decode(e, tokens) for e in two]
    assert all(torch.equal(a, b) for a, b in zip(*before)) and two[0].step_fn.resident._tiles is two[1].step_fn.resident._tiles is not None      # (once per model)
    w = m[1].blocks[1].feed_forward
    with torch.no_grad():
        w.w_down.mul_(0.5), w.w_gate.neg_()
    got = [decode(e, tokens) for e in two]      # (captured steps, replayed)
    assert all(torch.equal(a, b) for a, b in zip(*got)) and not torch.equal(got[0][0], before[0][0])
    other = model(*shape, "bfloat16")
    with torch.no_grad():
        other[1].blocks[1].feed_forward.w_down.mul_(0.5), other[1].blocks[1].feed_forward.w_gate.neg_()
    fresh = engine(other, rows, max(lengths) + 12, "bfloat16")
    stand(fresh, lengths, 1)
    first = decode(fresh, tokens[:1])
    late = engine(m, rows, max(lengths) + 12, "bfloat16")
    stand(late, lengths, 1)
    assert torch.equal(decode(late, tokens[:1])[0], first[0])


@pytest.mark.gpu
def test_nothing_is_laid_out_before_a_step_of_more_than_sixteen_rows():
    from test_resident_gpu import decode, engine, model, stand
    m = model(256, 4, 1, 512, "bfloat16")
    size = m[1].weight_bytes()
    e = engine(m, 17, 100, "bfloat16")
    stand(e, [5] * 17, 1)
    decode(e, [[1] * 16])
    assert m[1].tiles is None and m[1].weight_bytes() == size
    decode(e, [[1] * 17])
    assert m[1].weight_bytes() == size + 3 * 256 * 512 * 2 * len(m[1].order)


def steps_of(e, rows, launches):
    from test_resident_gpu import decode, stand
    stand(e, [5 + i for i in range(rows)], 1)
    del launches[:]
    out = decode(e, np.random.default_rng(rows).integers(0, 500, (3, rows)).tolist())
    assert set(launches) <= {rows} and e.step_fn.graph_replays + len(launches) >= 3      # (all layers in one launch)
    return out


@pytest.fixture
def launches(monkeypatch):
    from alofa_amd import ops
    made, one_launch = [], ops.decode_resident
    monkeypatch.setattr(ops, "decode_resident", lambda hidden, *a, **how: (made.append(hidden.shape[0]), one_launch(hidden, *a, **how))[1])
    return made


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rows", [((256, 4, 1, 512), 17), ((320, 5, 5, 768), 30), ((896, 14, 2, 4864), 33), ((896, 14, 2, 4864), 64), ((1024, 16, 2, 2304), 20)])
@pytest.mark.parametrize("why", ["no memory", "little room", "writes are not counted"])
def test_matrices_are_read_as_they_are_where_no_tiles_are(shape, rows, why, monkeypatch, launches):
    """One launch for all layers either way, and the same bits."""
    from alofa_amd import ops
    from test_resident_gpu import engine, model
    want = steps_of(engine(model(*shape, "bfloat16"), rows, 200, "bfloat16"), rows, launches)

    def none(*a):
        raise torch.cuda.OutOfMemoryError("no memory")
    if why == "no memory":
        monkeypatch.setattr(ops, "in_tiles", none)
    elif why == "little room":
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (0, 1 << 38)), monkeypatch.setattr(torch.cuda, "memory_reserved", lambda *a: torch.cuda.memory_allocated(*a))
    with torch.inference_mode(why == "writes are not counted"):
        m = model(*shape, "bfloat16")
    assert m[1].blocks[0].feed_forward.w_down.is_inference() == (why == "writes are not counted")
    e = engine(m, rows, 200, "bfloat16")
    got = steps_of(e, rows, launches)
    assert m[1].tiles is None and all(torch.equal(a, b) for a, b in zip(want, got))
    if why == "writes are not counted":      # (such a write is seen)
        from test_resident_gpu import decode
        with torch.inference_mode():
            m[1].blocks[0].feed_forward.w_down.neg_()
        assert not torch.equal(decode(e, [[1] * rows])[0], got[0])


@pytest.mark.gpu
def test_writes_that_are_not_counted_and_said(launches):
    """Through ``.data``: seen by steps of up to sixteen rows at once, by steps of more behind ``weights_written``."""
    from test_resident_gpu import engine, model
    m = model(256, 4, 1, 512, "bfloat16")
    e = engine(m, 20, 200, "bfloat16")
    before = steps_of(e, 20, launches)
    for i in range(20):
        e.cache.free(i)
    m[1].blocks[1].feed_forward.w_gate.data.neg_(), m[1].blocks[2].feed_forward.w_down.data.mul_(0.5)
    m[1].weights_written()
    got = steps_of(e, 20, launches)
    other = model(256, 4, 1, 512, "bfloat16")
    with torch.no_grad():
        other[1].blocks[1].feed_forward.w_gate.neg_(), other[1].blocks[2].feed_forward.w_down.mul_(0.5)
    want = steps_of(engine(other, 20, 200, "bfloat16"), 20, launches)
    assert all(torch.equal(a, b) for a, b in zip(want, got)) and not torch.equal(before[0], got[0])
