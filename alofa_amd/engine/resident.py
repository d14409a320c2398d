"""Decode steps whose layers run in one launch (csrc/decode_resident.hip, and csrc/decode_groups.hip for more
than 16 rows): what the launch needs beside the step's own tensors, kept by a step
function: the table of the layers' matrices and caches, an area of memory that the launch's blocks exchange values in, and a word that the
kernel sets if it gives a wait up."""
from __future__ import annotations

import collections
import contextlib
import fcntl
import os
import tempfile
import threading
import weakref
from typing import Optional

import torch

from .. import ops
from ..errors import AlofaError
from ..parts.attention import GQAAttention
from ..parts.block import PreNormBlock
from ..parts.feed_forward import SwiGLU


class _Area:
    """Memory that the blocks of a launch exchange values in, and the pinned word that the kernel sets if it gives a wait up."""

    def __init__(self):
        self.failed = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        self.address = ops.resident_area()


class _Areas:
    """Areas that step functions of this process have given back. They are never freed (uncached device memory must not be), so there are never
    more of them than step functions lived at one time. One that changes hands has no launch in flight: the taker waits for the device first. One
    whose owner failed is cleared then: the word that stops its launches is still set, and its counter and its values may not belong together."""

    def __init__(self):
        # device -> areas. No lock: ``give_back`` runs wherever the garbage collector does, in the middle of a ``take`` or of another ``give_back`` of the same
        # thread too (a deque's own operations are whole ones)
        self._idle: dict = {}

    def _of(self, device: torch.device) -> collections.deque:
        return self._idle.setdefault(device.index, collections.deque())

    def take(self, device: torch.device) -> _Area:
        try:
            area = self._of(device).pop()
        except IndexError:
            area = None
        with torch.cuda.device(device):
            if area is None:
                return _Area()
            torch.cuda.synchronize(device)
            if area.failed.item():
                ops.clear_resident_area(area.address)
                area.failed.zero_()
        return area

    def give_back(self, device: torch.device, area: _Area) -> None:
        self._of(device).append(area)


_areas = _Areas()


class _Seats:
    """Which processes run such launches on a GPU: at most two, as many as fit on it at once (a third's blocks and theirs could keep one another waiting). A process
    holds a lock on one of two files from its first such step function on until it ends, whichever way. Without one of them, or where the files cannot be had, steps
    run kernel by kernel. (Processes that do not share the folder do not know of one another: there ``ALOFA_ONE_LAUNCH=0`` in all but two.)"""

    def __init__(self, folder: Optional[str] = None):
        self.folder = folder or tempfile.gettempdir()
        self._lock = threading.Lock()
        self._held: dict = {}      # (process, GPU) -> the open file whose lock this process has

    @staticmethod
    def _open(path: str) -> Optional[int]:
        flags = os.O_RDWR | os.O_CLOEXEC | os.O_NOFOLLOW
        for _ in range(2):      # (a file that is there is opened as it is: a sticky folder refuses O_CREAT for another user's)
            try:
                return os.open(path, flags)
            except FileNotFoundError:
                pass
            except OSError:
                return None
            try:
                fd = os.open(path, flags | os.O_CREAT | os.O_EXCL, 0o666)
                os.fchmod(fd, 0o666)
                return fd
            except FileExistsError:
                pass
            except OSError:
                return None
        return None

    def take(self, gpu: str) -> bool:
        with self._lock:
            key = (os.getpid(), gpu)      # (a fork has the open file, but not the lock)
            if key in self._held:
                return True
            for n in range(2):
                fd = self._open(os.path.join(self.folder, f"alofa_amd-one-launch-{gpu}-{n}.lock"))
                if fd is None:
                    continue
                try:
                    fcntl.lockf(fd, fcntl.LOCK_EX | fcntl.LOCK_NB)
                except OSError:
                    os.close(fd)
                    continue
                self._held[key] = fd
                return True
            return False


_seats = _Seats()


class _Turns:
    """Launches of one GPU's steps go one after the other, whichever threads and streams of this process they come from: a launch's blocks hold half of
    every compute unit until all of them have come, so that two launches fit (another process may have the other half), a third may not. A launch on another stream than
    the last one's waits for what that stream had been given; on the same stream nothing is added. Held for the launch alone: not while a step is laid out or captured, and not while it runs."""

    def __init__(self, device: torch.device):
        self._device, self._lock = device, threading.Lock()
        self._last: Optional[torch.cuda.Stream] = None      # the stream of the last launch

    def __enter__(self):
        self._lock.acquire()
        try:
            here, last = torch.cuda.current_stream(self._device), self._last
            if last is not None and last != here:
                reached = torch.cuda.Event()
                reached.record(last)
                here.wait_event(reached)
            self._last = here
        except BaseException:
            self._lock.release()
            raise
        return self

    def __exit__(self, *exc):
        self._lock.release()
        return False


_turns: dict = {}      # GPU -> its launches' turns


class _Tiles:
    """Copies of a model's gate, up and down matrices as more than sixteen rows read them (``ops.in_tiles``): made once per model, for all its step functions, and again where the matrices have been
    written since: as far as torch counts the writes, and where ``Model.weights_written`` says so."""
    ROOM = 2      # times their size that must be free before they are laid out: the rest is what a service's scratch grows into

    def __init__(self, model, sources: list):
        self._model, self._sources, self._lock = weakref.ref(model), sources, threading.Lock()
        versions = self._now()
        self.copies = [ops.in_tiles(w) for w in sources]
        torch.cuda.current_stream(sources[0].device).synchronize()      # (steps on other streams read them too)
        self._versions = versions

    def _now(self) -> list:
        model = self._model()
        return [None if model is None else model.written, *(w._version for w in self._sources)]

    def bytes(self) -> int:
        return sum(t.numel() * t.element_size() for t in self.copies)

    def follow(self) -> None:
        if self._now() == self._versions:
            return
        with self._lock:
            now = self._now()
            if now != self._versions:
                device = self._sources[0].device
                torch.cuda.synchronize(device)      # (steps of other streams that are on their way read what is there now)
                for w, to in zip(self._sources, self.copies):
                    ops.in_tiles(w, to)
                torch.cuda.current_stream(device).synchronize()
                self._versions = now

    @staticmethod
    def of(model, sources: list) -> Optional["_Tiles"]:
        """None where the matrices are read as they are instead: where torch does not count the writes to them (inference tensors), or there is no memory to spare."""
        with _laying_out:
            have = model.tiles
            if have is None or len(have._sources) != len(sources) or any(a is not b for a, b in zip(have._sources, sources)):
                if any(w.is_inference() for w in sources):
                    return None
                device = sources[0].device
                free = torch.cuda.mem_get_info(device)[0] + torch.cuda.memory_reserved(device) - torch.cuda.memory_allocated(device)
                if free < _Tiles.ROOM * sum(w.numel() * w.element_size() for w in sources):
                    return None
                try:
                    model.tiles = _Tiles(model, sources)
                except torch.cuda.OutOfMemoryError:
                    return None
            return model.tiles


_laying_out = threading.Lock()


class ResidentLayers:
    """All layers of ``model`` over ``cache`` as one launch, for steps of at most ``MOST_ROWS`` rows of one new token each."""
    MOST_ROWS = most_rows = 16      # (``most_rows``: of this model, up to 64: csrc/decode_groups.hip)
    MOST_LAYERS = 64      # whose addresses the kernel keeps at hand
    # (rows x key heads below, keys that the longest request sees): the launch cuts a row and key head's keys into sixteen parts, the kernels one by one into as many as the chip has
    # compute units for, up to 64. us a step, one launch / kernel by kernel: one row, two key heads of the 0.5B sizes, 16,000 keys 629 / 764, 31,000 813 / 779; one row and key head, 256
    # wide (24 layers), 15,000 491 / 542, 31,000 668 / 562, 512 wide (16) 344 / 382 and 469 / 398; three key heads, 576 wide (30), 682 / 793 and 919 / 820; rows x key heads of four or five,
    # 31,000 keys: 840 / 846, 299 / 297, 802 / 804, 560 / 573; of eight 924 / 1,022; of sixteen 1,076 / 1,335, 484 / 617. Even at 20,000 to 28,000 below four, at 30,000 from there on.
    MOST_KEYS = ((4, 20000), (16, 28000))
    # Groups (more than MOST_ROWS rows) deal their blocks to their rows' key heads, a block at least to each. Where a row of more than LONG_KEYS keys is left with one block a key head, the
    # layer waits for that block while others idle. us a step of 6 layers, kernel by kernel / groups, blocks with keys of 64: four key heads, 33 rows of 16,000 keys (36) 1,017 / 1,111, 48
    # (48) 1,126 / 1,196, 56 (56) 1,270 / 1,209; 24 of 14,000 beside 24 short ones 906 / 962; 28 beside five, two blocks to each, 926 / 700; three key heads, 48 of 24,000 (36) 1,338 / 1,561,
    # 40 (30, twice) 1,055 / 971, 64 of 14,000 (48) 1,017 / 1,088. So groups where every long row has two blocks a key head, or where such rows fill thirteen of sixteen blocks (52 rows of
    # 14,000 with four key heads 1,090 / 1,076). Rows of 4,000 gain 1.08 to 1.24 throughout, of 8,000 0.97 to 1.19.
    LONG_KEYS, BLOCKS = 7000, 256      # (blocks of a launch)

    @classmethod
    def of(cls, model, cache) -> Optional["ResidentLayers"]:
        """None where the model's layers are not what the kernel runs: pre-norm blocks of grouped-query attention over its own cache of every token (rotary, no
        output bias) and a silu-gated feed-forward, all alike, sizes that fit a block's registers, bfloat16; or where ``ALOFA_ONE_LAUNCH=0`` or other processes say no."""
        rt, order = model.rt, model.order
        if os.environ.get("ALOFA_ONE_LAUNCH", "1") == "0" or rt.exact or rt.dtype is not torch.bfloat16 or model.streams or model.joins or not 0 < len(order) <= cls.MOST_LAYERS:
            return None
        blocks = [model.blocks[e.layer] for e in order]
        if any(e.cache_of is not None or e.join is not None for e in order) or any(type(b) is not PreNormBlock for b in blocks):
            return None
        first = blocks[0]
        for i, b in enumerate(blocks):
            m, f = b.mixer, b.feed_forward
            if type(m) is not GQAAttention or type(f) is not SwiGLU or f.activation != "silu" or m.window is not None or m.b_o is not None:
                return None
            if any(n.as_rmsnorm() is None for n in b.norms) or m.position.table(1) is None or cache.group_of_entry.get((i, 0)) is None:
                return None
            same = [(x.mixer.heads, x.mixer.kv_heads, x.mixer.d, x.mixer.scale, x.mixer.b_qkv is None, x.mixer.hidden, x.feed_forward.intermediate, tuple(n.as_rmsnorm()[1] for n in x.norms),
                     x.mixer.position.table(1)[0].data_ptr()) for x in (first, b)]
            if same[0] != same[1] or cache.group_of_entry[(i, 0)] != cache.group_of_entry[(0, 0)]:
                return None
        m = first.mixer
        if not ops.resident_takes(m.hidden, first.feed_forward.intermediate, m.heads, m.kv_heads, m.d, cache.block_size):
            return None
        tables = [cls._tensors(b, cache.tensors[(i, 0)]) for i, b in enumerate(blocks)]
        if not all(cls._reads(m, first.feed_forward.intermediate, t) for t in tables):
            return None
        device = rt.device if rt.device.index is not None else torch.device(rt.device.type, torch.cuda.current_device())      # (by number, so that all of a GPU's launches meet)
        if not _seats.take(str(torch.cuda.get_device_properties(device).uuid)):
            return None
        try:
            area = _areas.take(device)
        except (AlofaError, RuntimeError):      # (no memory for one: the kernels one by one need none)
            return None
        return cls(model, blocks, cache, device, tables, area)

    @staticmethod
    def _tensors(b, kv: dict) -> list:
        """What the kernel reads of a layer, in its order: matrices and bias, norms, caches."""
        return [b.mixer.w_qkv, b.mixer.b_qkv, b.mixer.w_o, b.feed_forward.w_gate, b.feed_forward.w_up, b.feed_forward.w_down,
                b.norms[0].as_rmsnorm()[0], b.norms[1].as_rmsnorm()[0], kv["k"], kv["v"]]

    @staticmethod
    def _reads(m, intermediate: int, tensors: list) -> bool:
        """Whether a layer's tensors are what the kernel takes them for: matrices are kept in the type they were stored in and where their owner has them, so they may
        be float32, or begin where no load of sixteen bytes can (the products one by one take those too)."""
        qkv, out, h = (m.heads + 2 * m.kv_heads) * m.d, m.heads * m.d, m.hidden
        shapes = [(qkv, h), (qkv,), (h, out), (intermediate, h), (intermediate, h), (h, intermediate), (h,), (h,), None, None]
        for t, shape in zip(tensors, shapes):
            if t is None:      # (no bias)
                continue
            dtype = torch.float32 if shape is not None and len(shape) == 1 else torch.bfloat16
            if not t.is_cuda or t.dtype is not dtype or not t.is_contiguous() or t.data_ptr() % 16 or (shape is not None and tuple(t.shape) != shape):
                return False
        return True

    def __init__(self, model, blocks: list, cache, device, tables: list, area: "_Area"):
        self.device, self.area = device, area
        weakref.finalize(self, _areas.give_back, device, area)
        m = blocks[0].mixer
        self.heads, self.kv_heads, self.d, self.scale, self.position = m.heads, m.kv_heads, m.d, m.scale, m.position
        self.hidden, self.intermediate, self.biased = m.hidden, blocks[0].feed_forward.intermediate, m.b_qkv is not None
        self.most_rows = ops.resident_rows(self.hidden, self.intermediate, self.heads, self.kv_heads)
        self.eps = tuple(float(n.as_rmsnorm()[1]) for n in blocks[0].norms)
        self.page, self.group = cache.block_size, cache.group_of_entry[(0, 0)]
        for t in tables:
            ops.check_caches(t[-2], t[-1], self.kv_heads, self.d)
        self._tables = tables      # (kept: the table on the GPU holds their addresses)
        self._model, self._tiles, self._asked, self._addresses = model, None, False, [[0 if t is None else t.data_ptr() for t in ts] for ts in tables]
        # the layers' addresses on the GPU, and behind them, for more rows than sixteen, those with gate, up and down in tiles (once these are laid out). Launches read it whenever they run, captured ones as
        # long as their graphs live: it is made once and never moves
        self._table = torch.tensor([self._addresses] * 2 if self.most_rows > self.MOST_ROWS else self._addresses, dtype=torch.int64, device=device)
        self._few = self._table if self._table.dim() == 2 else self._table[0]
        self.failed = area.failed
        self._failed = self.failed.numpy()
        self.turn = _turns.setdefault(device.index, _Turns(device))      # what a launch, or a replay of one, goes within

    def takes(self, ctx, rows: int) -> bool:
        """Whether this step runs in one launch: one new token for each of few requests, and keys that it is the faster one for."""
        if rows > self.most_rows or ctx.max_q_len != 1 or len(ctx.spans) != rows:
            return False
        if rows > self.MOST_ROWS and ctx.longest > self.LONG_KEYS:
            groups = 2 if rows <= 2 * self.MOST_ROWS else 4
            blocks = self.BLOCKS // groups
            pairs, long = (-(-n // groups) * self.kv_heads for n in (rows, sum(s.pos0 + s.n > self.LONG_KEYS for s in ctx.spans)))
            if pairs + long > blocks and 16 * long < 13 * blocks:
                return False
        return ctx.longest <= next((keys for below, keys in self.MOST_KEYS if rows * self.kv_heads < below), ctx.longest)

    @property
    def layers(self) -> torch.Tensor:
        """The layers' addresses as ``ops.decode_resident`` takes them. Gate, up and down in tiles, which more rows than sixteen read where there is room for them, are laid out when they are first asked for."""
        if not self._asked and self.most_rows > self.MOST_ROWS and not torch.cuda.is_current_stream_capturing():
            tiles = _Tiles.of(self._model, [w for ts in self._tables for w in ts[3:6]])
            if tiles is not None:
                places = [t.data_ptr() for t in tiles.copies]
                self._table[1].copy_(torch.tensor([[*a[:3], *places[3 * i:3 * i + 3], *a[6:]] for i, a in enumerate(self._addresses)], dtype=torch.int64))
            self._tiles, self._asked = tiles, True      # (once: captured steps of more rows are of one kind)
        return self._table if self._tiles is not None or self._table.dim() == 2 else self._table[0]

    def ready(self, rows: int) -> None:
        """In front of a step that is taken, or a replay of one: what is laid out of the matrices is what they hold."""
        if rows > self.MOST_ROWS:
            self.layers
            if self._tiles is not None and not torch.cuda.is_current_stream_capturing():
                self._tiles.follow()

    def gave_up(self) -> bool:
        return bool(self._failed[0])

    def forward(self, ctx, hidden: torch.Tensor) -> None:
        cos, sin = self.position.table(ctx.n_positions)
        with contextlib.nullcontext() if torch.cuda.is_current_stream_capturing() else self.turn:      # (one that is captured takes its turn at every replay)
            ops.decode_resident(hidden, self.layers if hidden.shape[0] > self.MOST_ROWS else self._few, ctx.positions, ctx._tables[self.group], ctx._slots[self.group], cos, sin, self.area.address, self.failed, self.intermediate,
                                self.heads, self.kv_heads, self.d, self.page, self.biased, self.scale, self.eps)
