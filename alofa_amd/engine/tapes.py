"""Layers that are alike, in steps that run kernel by kernel: the launches of one are noted as it runs and made again for the others with their
tensors in its tensors' places, without a way through Python for every launch.

A step's layers launch the same kernels on the same buffers and differ in their own matrices, vectors and caches only. A launch takes the host
7.4 us by way of the parts and 3.6 so: three prompts of 5 to 33 tokens at the 0.5B sizes (24 layers, 172 launches), which wait for the host, 1,445 and 1,219 us a step, of which it
is the kernels then that take the time."""
from __future__ import annotations

import operator
import os
from typing import Optional

import numpy as np
import torch

from .. import ops
from ..parts.base import Part, repeats

SWITCHED_ON = os.environ.get("ALOFA_TAPES", "1") != "0"      # 0 (for measurements): every layer goes through its parts


class _Walk:
    """What makes up a block, in a fixed order: ``seen``, for comparison, and the block's ``tensors``. ``refs``: where its tensors, parts and containers were found, (container, key, value);
    ``plain``: the same of numbers and names."""

    def __init__(self, block):
        self.seen, self.tensors, self.refs, self.plain, self._parts = [type(block)], [], [], [], {}
        self._part(block)

    def _part(self, part) -> None:
        if id(part) in self._parts:
            self.seen.append(self._parts[id(part)])
            return
        self._parts[id(part)] = len(self._parts)
        own = vars(part)
        for name in sorted(own):
            if name not in ("rt", "spec", "layer"):      # (the runtime is the model's; the descriptions name tensors: what the parts made of them is compared)
                self._value(own, name)

    def _value(self, within, key) -> None:
        v = within[key]
        self.seen.append((key, type(v)))
        if v is None or isinstance(v, (bool, int, float, str, bytes, torch.dtype, torch.device)):
            self.seen.append(v)
            if not isinstance(within, tuple):
                self.plain.append((within, key, v))
            return
        if not isinstance(within, tuple):
            self.refs.append((within, key, v))
        if isinstance(v, torch.Tensor):
            self.tensors.append(v)
            self.seen.append((tuple(v.shape), v.stride(), v.dtype, str(v.device), v.data_ptr() % 64))
        elif isinstance(v, Part):
            self._part(v)
        elif isinstance(v, (list, tuple)):
            self.seen.append(len(v))
            for k in range(len(v)):
                self._value(v, k)
        elif type(v) is dict:
            self.seen.append(len(v))
            for k in sorted(v, key=repr):
                self._value(v, k)
        elif isinstance(v, np.ndarray):
            self.seen.append((v.shape, v.dtype.str, v.tobytes()))
        else:
            self.seen.append(id(v))      # (alike is the very same one, which ``refs`` holds)


def _stand(within, keys, values) -> bool:
    """Whether within[i][keys[i]] is values[i] throughout."""
    try:
        return all(map(operator.is_, map(operator.getitem, within, keys), values))
    except (KeyError, IndexError):
        return False


class LayerTapes:
    """For a step function: which entries of the model's order are alike, and where their tensors lie."""

    @staticmethod
    def of(model, cache) -> Optional["LayerTapes"]:
        if not SWITCHED_ON or model.joins or model.streams or not any(repeats(b) for b in model.blocks):
            return None
        tapes = LayerTapes(model, cache)
        return tapes if tapes.source else None

    def __init__(self, model, cache):
        walks = model.descriptions      # (a step function before this one may have looked: 2 ms for 24 layers, a tenth of it to see whether they are what they were)
        if walks is None or not all(_stand(*zip(*w.refs, *w.plain)) for w in walks):
            walks = model.descriptions = [_Walk(b) for b in model.blocks]
        owners = model.cache_owners()
        layers = [e.layer for e in model.order]
        kinds, self._tensors = [], []      # (the tensors are held: their addresses stay theirs)
        for i, layer in enumerate(layers):
            if not repeats(model.blocks[layer]) or owners.get((i, 0)) != (i, 0) or i + 1 == len(layers):
                kinds.append(None), self._tensors.append(None)
                continue
            # (a block is handed the norm that the next one starts with; which tensors of either a launch takes does not matter here)
            mine, next_one = walks[layer], walks[layers[i + 1]]
            caches = [t for _, t in sorted(cache.tensors[(i, 0)].items())]
            tensors = [*mine.tensors, *next_one.tensors, *caches]
            places = [t.data_ptr() for t in tensors]
            # (last: which of them are one and the same)
            kinds.append((mine.seen, next_one.seen, cache.group_of_entry[(i, 0)], tuple((t.shape, t.stride(), t.dtype, t.data_ptr() % 64) for t in caches),
                          None if len(set(places)) == len(places) else tuple(places.index(p) for p in places)))
            self._tensors.append(tensors)
        # entry -> the first entry of its run of alike ones (entries behind the first in the order: what stands in front of them is alike too)
        self.source, first = {}, None
        for i in range(1, len(layers)):
            if kinds[i] is None or first is None or kinds[i] != kinds[first]:
                first = i if kinds[i] is not None else None
            else:
                self.source[i] = first
        self.sources = set(self.source.values())
        self._tensors = [t if i in self.source or i in self.sources else None for i, t in enumerate(self._tensors)]
        self._addresses = [None if t is None else tuple(x.data_ptr() for x in t) for t in self._tensors]
        self._bytes = {i: tuple(x.numel() * x.element_size() for x in self._tensors[i]) for i in self.sources}

        # where what was looked at was found, to be looked at again before a step
        used = {layers[i + more] for i in {*self.source, *self.sources} for more in (0, 1)}
        refs = [r for layer in sorted(used) for r in walks[layer].refs]
        self._within, self._keys, self._values = ([r[k] for r in refs] for k in range(3))

    def stand(self) -> bool:
        """Whether the parts still hold the tensors and parts that were compared (11 us for 24 layers, in a step that takes the host a millisecond)."""
        return _stand(self._within, self._keys, self._values)

    def addresses(self, entry: int) -> tuple:
        return self._addresses[entry]

    def note(self, entry: int) -> ops.tape_calls:
        return ops.tape_calls(tuple(zip(self._addresses[entry], self._bytes[entry])))
