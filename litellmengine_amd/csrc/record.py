"""The launches of one layer, kept while it runs, and launched again for the layers behind it that are alike.

A launch costs the host about 3 us in the runtime and 5 to 17 us in Python: checks, the choice of a kernel, the result's
memory.  Layers that differ in nothing but where their weights and their cache lie get the same launches with other addresses, so
a step pays for the rest once: while a layer runs, `HipOps` keeps what it launches (`LaunchRecord`), and a `Replay` launches it
again with another layer's operands in their places.  Both live inside one forward pass; nothing of them is kept for the next.
Host time of a step of 28 layers 1024 wide, 8 and 280 tokens: 1.96 -> 1.15 and 3.23 -> 2.07 ms."""
from __future__ import annotations

import bisect
import ctypes
from typing import Dict, List, Optional, Sequence

import torch


class LaunchRecord:
    """What was launched on `stream`, in order, and every tensor that was made for it (kept alive)."""

    def __init__(self, stream: int):
        self.stream = stream
        self.calls: List[tuple] = []  # (function, name, arguments), or for a library product (None, take, x, weight, result)
        self.made: List[torch.Tensor] = []
        self.whole = True  # everything was launched on that stream

    def launch(self, fn, lib: str, name: str, args, stream: int) -> None:
        self.whole = self.whole and stream == self.stream
        self.calls.append((fn, (lib, name), args))

    def product(self, take, x, weight, result) -> None:
        """`take(x, weight, out)`: the library's product, into a tensor that is there."""
        self.calls.append((None, take, x, weight, result))
        self.made += [x, result]


class Replay:
    """A record's launches for operands that lie elsewhere.  `operands`: the recorded layer's tensors that differ from layer
    to layer; `given`: what it took over from the layer before; `left`: what it left for the next one, which then is that
    layer's `given`, and is written in the place where the recorded layer wrote it."""

    def __init__(self, record: LaunchRecord, operands: Sequence[torch.Tensor], given: Sequence[torch.Tensor], left: Sequence[torch.Tensor]):
        self.ok = False
        places: Dict[int, int] = {}
        for i, t in enumerate(operands):
            if places.setdefault(t.data_ptr(), i) != i:
                return  # (one tensor in two places: which of them a launch means cannot be told)
        if not record.whole or len(given) != len(left) or any(a.shape != b.shape or a.dtype != b.dtype for a, b in zip(given, left)):
            return
        over = {t.data_ptr(): u.data_ptr() for t, u in zip(given, left)}
        if len(over) != len(given) or any(p in places for p in over) or any(u in places or u in over for u in over.values()):
            return
        spans = sorted((t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for t in (*operands, *given))
        starts = [a for a, _ in spans]
        written = set(over.values())
        self.calls, last_given, first_left = [], -1, len(record.calls)
        for n, call in enumerate(record.calls):
            if call[0] is None:
                _, take, x, weight, result = call
                i = places.get(weight.data_ptr())
                if i is None or any(t.data_ptr() in over or t.data_ptr() in places for t in (x, result)):
                    return
                if x.data_ptr() in written or result.data_ptr() in written:
                    first_left = min(first_left, n)
                self.calls.append((None, take, x, i, result))
                continue
            fn, name, args = call
            args, patches = list(args), []
            for k, (kind, p) in enumerate(zip(fn.argtypes, args)):
                if kind is not ctypes.c_void_p or not p:
                    continue
                if p in places:
                    patches.append((k, places[p]))
                elif p in over:
                    args[k], last_given = over[p], n
                elif p in written:
                    first_left = min(first_left, n)
                else:
                    at = bisect.bisect_right(starts, p) - 1
                    if at >= 0 and p < spans[at][1]:
                        return  # (inside an operand, or inside what was taken over)
            self.calls.append((fn, name, args + [record.stream], tuple(patches), None))
        # what a layer takes over has been read before the same memory is written for the next one
        self.ok = last_given < first_left

    def run(self, operands: Sequence[torch.Tensor], addresses: Sequence[int]) -> Optional[tuple]:
        """None, or (library, function, code) of a launch that failed."""
        for fn, name, args, patches, result in self.calls:
            if fn is None:
                name(args, operands[patches], result)  # (take(x, weight, out))
                continue
            for k, i in patches:
                args[k] = addresses[i]
            code = fn(*args)
            if code:
                return name + (code,)
        return None


def operand_kinds(tensors: Sequence[torch.Tensor]) -> list:
    """What a launch's choice of a kernel and its checks see of its operands: sizes, types and whether they begin at 16 bytes."""
    return [(t.shape, t.dtype, t.data_ptr() & 15) for t in tensors]


def addresses_of(tensors: Sequence[torch.Tensor], kinds: list) -> Optional[List[int]]:
    """Where tensors of these kinds lie; None where one is of another kind, or where no launch would take it."""
    out = []
    for t, (shape, dtype, low) in zip(tensors, kinds):
        p = t.data_ptr()
        if t.shape != shape or t.dtype is not dtype or p & 15 != low or not t.is_contiguous() or not t.is_cuda:
            return None
        out.append(p)
    return out if len(tensors) == len(kinds) else None
