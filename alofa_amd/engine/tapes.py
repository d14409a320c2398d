"""Layers that are alike, in steps that run kernel by kernel: the launches of one are noted as it runs and made again for the others with their
tensors in its tensors' places, without a way through Python for every launch.

A step's layers launch the same kernels on the same buffers and differ in their own matrices, vectors and caches only. A launch takes the host
7.4 us by way of the parts and 3.6 so: three prompts of 5 to 33 tokens at the 0.5B sizes (24 layers, 172 launches), which wait for the host, 1,445 and 1,219 us a step, of which it
is the kernels then that take the time."""
from __future__ import annotations

import os
from typing import Optional

import torch

from .. import ops
from ..parts.base import Part

SWITCHED_ON = os.environ.get("ALOFA_TAPES", "1") != "0"      # 0 (for measurements): every layer goes through its parts


def _walk(part, tensors: list, seen: list) -> None:
    """The tensors of a part and of the parts within it, and what else makes up its behaviour, in a fixed order."""
    for name, v in sorted(vars(part).items()):
        if name in ("rt", "spec", "layer"):      # (the runtime is the model's; the descriptions name tensors: what the parts made of them is compared)
            continue
        for x in v if isinstance(v, (list, tuple)) else [v]:
            if isinstance(x, torch.Tensor):
                tensors.append(x)
                seen.append((name, tuple(x.shape), x.stride(), x.dtype, str(x.device), x.data_ptr() % 64))
            elif isinstance(x, Part):
                seen.append((name, type(x)))
                _walk(x, tensors, seen)
            else:
                seen.append((name, repr(x)))


def _describe(block) -> tuple:
    """(what makes up the block, its tensors)"""
    tensors, seen = [], [type(block)]
    _walk(block, tensors, seen)
    return tuple(seen), tensors


class LayerTapes:
    """For a step function: which entries of the model's order are alike, and where their tensors lie."""

    @staticmethod
    def of(model, cache) -> Optional["LayerTapes"]:
        if not SWITCHED_ON or model.joins or model.streams or not any(getattr(b, "repeatable", False) for b in model.blocks):
            return None
        tapes = LayerTapes(model, cache)
        return tapes if tapes.source else None

    def __init__(self, model, cache):
        if model.descriptions is None:      # (once per model: every step function of it asks)
            model.descriptions = [_describe(b) for b in model.blocks]
        owners = model.cache_owners()
        layers = [e.layer for e in model.order]
        kinds, self._tensors = [], []      # (the tensors are held: their addresses stay theirs)
        for i, layer in enumerate(layers):
            if not getattr(model.blocks[layer], "repeatable", False) or owners.get((i, 0)) != (i, 0) or i + 1 == len(layers):
                kinds.append(None), self._tensors.append(None)
                continue
            # (a block is handed the norm that the next one starts with; which tensors of either a launch takes does not matter here)
            (mine, tensors), (next_one, its_tensors) = model.descriptions[layer], model.descriptions[layers[i + 1]]
            caches = [t for _, t in sorted(cache.tensors[(i, 0)].items())]
            tensors = [*tensors, *its_tensors, *caches]
            places = [t.data_ptr() for t in tensors]
            # (last: which of them are one and the same)
            kinds.append((mine, next_one, cache.group_of_entry[(i, 0)], tuple((t.shape, t.stride(), t.dtype, t.data_ptr() % 64) for t in caches),
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

    def addresses(self, entry: int) -> tuple:
        return self._addresses[entry]

    def note(self, entry: int) -> ops.tape_calls:
        return ops.tape_calls(tuple(zip(self._addresses[entry], self._bytes[entry])))
