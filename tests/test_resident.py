"""Decode steps in one launch: what lies around the launch, without a GPU."""
import gc
import os
import signal
import threading
import weakref
from types import SimpleNamespace

import pytest
import torch

from alofa_amd.engine.resident import ResidentLayers, _Areas, _Seats


def another(folder):
    """Another process that asks for a seat and lives until ``end``: (process, what ends it, whether it has one)."""
    (said, say), (told, tell) = os.pipe(), os.pipe()
    pid = os.fork()
    if pid == 0:
        try:
            os.close(tell)
            os.write(say, b"1" if _Seats(str(folder)).take("gpu") else b"0")
            os.read(told, 1)
        finally:
            os._exit(0)
    os.close(say), os.close(told)
    has = os.read(said, 1) == b"1"
    os.close(said)
    return (pid, tell), has


def end(process, how=None):
    pid, tell = process
    if how:
        os.kill(pid, how)
    else:
        os.write(tell, b".")      # (closing it would not do: processes forked later have it open too)
    os.close(tell)
    os.waitpid(pid, 0)


def test_two_processes_have_a_seat_on_a_gpu_and_a_third_has_none(tmp_path):
    mine = _Seats(str(tmp_path))
    assert mine.take("gpu") and mine.take("gpu")      # (one seat, however often it is asked for)
    second, has = another(tmp_path)
    assert has
    third, has = another(tmp_path)
    assert not has
    end(third)
    assert mine.take("another gpu")
    end(second)      # its seat is free again
    fourth, has = another(tmp_path)
    assert has
    end(fourth, signal.SIGKILL)      # whichever way a process ends
    fifth, has = another(tmp_path)
    assert has
    end(fifth)


def test_a_fork_does_not_have_its_parents_seat(tmp_path):
    seats = _Seats(str(tmp_path))
    assert seats.take("gpu")
    other, has = another(tmp_path)
    assert has
    pid = os.fork()
    if pid == 0:
        os._exit(0 if not seats.take("gpu") else 1)
    assert os.waitpid(pid, 0)[1] == 0
    end(other)
    third, has = another(tmp_path)      # the parent's seat is still held: one was free
    assert has
    fourth, has = another(tmp_path)
    assert not has
    end(third), end(fourth)


def test_no_seat_where_the_files_cannot_be_had(tmp_path):
    assert not _Seats(str(tmp_path / "none")).take("gpu")
    for n in range(2):
        os.symlink("/dev/null", tmp_path / f"alofa_amd-one-launch-gpu-{n}.lock")
    assert not _Seats(str(tmp_path)).take("gpu")


def test_a_scope_of_one_thread_leaves_the_streams_of_others_alone(monkeypatch):
    """Two threads whose scopes overlap, neither within the other: each launches on its own stream inside and outside its scope."""
    from alofa_amd import ops
    current = threading.local()
    monkeypatch.setattr(ops.torch.cuda, "current_stream", lambda *a: SimpleNamespace(cuda_stream=current.stream))
    current.stream = 1
    entered, leave, seen = threading.Event(), threading.Event(), {}

    def other():
        current.stream = 2
        seen["before"] = ops._stream()
        with ops.stream_scope():
            entered.set()
            leave.wait(30)
            seen["within"] = ops._stream()
        seen["behind"] = ops._stream()
    with ops.stream_scope():
        t = threading.Thread(target=other)
        t.start()
        assert entered.wait(30)
        assert ops._stream() == 1
    assert ops._stream() == 1
    leave.set()
    t.join(30)
    assert seen == {"before": 2, "within": 2, "behind": 2}
    current.stream = 3
    assert ops._stream() == 3


def test_an_area_is_given_back_while_another_is_being_given_back():
    """By a finalizer that the collector runs in the middle of it, on the same thread."""
    areas, device = _Areas(), torch.device("cuda:0")

    class Collecting(dict):
        def setdefault(self, key, value):
            gc.collect()
            return super().setdefault(key, value)
    areas._idle = Collecting()

    class Owner:
        def __init__(self):
            self.me = self      # (goes only when the collector comes)
            weakref.finalize(self, areas.give_back, device, object())

    def work():
        gc.disable()
        Owner()
        areas.give_back(device, object())
    t = threading.Thread(target=work, daemon=True)
    try:
        t.start()
        t.join(10)
    finally:
        gc.enable()
    assert not t.is_alive()
    assert sum(len(a) for a in areas._idle.values()) == 2


def test_steps_of_few_rows_over_very_many_keys_are_left_to_the_kernels_one_by_one():
    layers = ResidentLayers.__new__(ResidentLayers)

    def takes(rows, kv_heads, longest, new=1):
        layers.kv_heads = kv_heads
        return layers.takes(SimpleNamespace(max_q_len=new, spans=[None] * rows, longest=longest), rows)
    assert takes(1, 2, 20000) and not takes(1, 2, 20001)
    assert takes(3, 1, 20000) and not takes(3, 1, 20001)
    assert takes(2, 2, 28000) and not takes(2, 2, 28001)
    assert takes(5, 3, 28000) and not takes(5, 3, 28001)
    assert takes(8, 2, 1000000) and takes(1, 16, 1000000) and takes(16, 1, 1000000)
    assert not takes(17, 1, 10) and not takes(1, 1, 10, new=2)


@pytest.mark.parametrize("kv_heads,long,short,taken", [
    (4, 33, 0, False), (4, 48, 0, False), (4, 52, 0, True), (4, 64, 0, True), (4, 24, 24, False), (4, 28, 5, True), (4, 0, 64, True),     # 64 blocks a group
    (3, 40, 0, True), (3, 48, 0, False), (3, 64, 0, False), (3, 28, 20, True), (2, 48, 0, True), (2, 64, 0, True), (1, 64, 0, True),
    (4, 32, 0, True), (8, 17, 0, False), (8, 28, 0, True), (8, 0, 17, True),     # 128
    (4, 16, 0, True),     # one group
])
def test_groups_where_long_rows_have_two_blocks_a_key_head(kv_heads, long, short, taken):
    rule = SimpleNamespace(MOST_ROWS=16, most_rows=64, kv_heads=kv_heads, MOST_KEYS=ResidentLayers.MOST_KEYS, LONG_KEYS=ResidentLayers.LONG_KEYS, BLOCKS=ResidentLayers.BLOCKS)
    keys = [ResidentLayers.LONG_KEYS + 1] * long + [ResidentLayers.LONG_KEYS] * short
    ctx = SimpleNamespace(max_q_len=1, longest=max(keys), spans=[SimpleNamespace(pos0=n - 1, n=1) for n in keys])
    assert ResidentLayers.takes(rule, ctx, len(keys)) is taken
