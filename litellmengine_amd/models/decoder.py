"""A decoder language model as data: an embedding, a set of blocks, the list
that says in which order they run (and with which cache), a final norm and an
output head.

The reference hard-wires embed -> layer 0..L-1 -> norm -> lm_head on all rows
(src/model/qwen3.cpp:1242-1278, :1501).  Here the order is a list of
`PlanEntry`: an entry may name a block that another entry names too (the
block's weights are then shared and it runs twice), and an entry may read the
cache that another entry writes instead of owning one.  The head runs on the
wanted rows only.
"""
from __future__ import annotations

import dataclasses
from typing import Dict, List, Optional, Sequence

import torch

from ..csrc.record import Replay, addresses_of, operand_kinds
from ..parts.base import Block, BuildContext, Carried, Injected, Norm, Normed, PartialSums, Prenormed, parts_as_written
from ..parts.embedding import Embedding
from ..parts.injection import PassVectors
from ..parts.linear import Linear
from ..weights.spec import TensorSpec


@dataclasses.dataclass(frozen=True)
class Inject:
    """What is added to the residual stream right before a plan entry's block: row `vector` of the model's
    pass vectors (None: none), and with `embedding` the embedding's rows once more."""

    vector: Optional[int] = None
    embedding: bool = False


@dataclasses.dataclass(frozen=True)
class PlanEntry:
    """One call of a block.  `cache` names the cache layer the mixer works on
    (default: one of its own, numbered like the entry); `writes=False` makes the
    entry a reader of a cache that an earlier entry fills; `inject` adds something to
    the stream ahead of the block."""

    block: int
    cache: Optional[int] = None
    writes: bool = True
    inject: Optional[Inject] = None


def looped_plan(blocks: int, start: int, stop: int, times: int, inject: bool = True) -> List[PlanEntry]:
    """Blocks start .. stop - 1 run `times` times in a row (each time with caches and states of their own), the
    others once.  Ahead of pass t the stream gets pass vector t, and from the second pass on also the embedding's rows
    (`inject=False`: nothing enters the stream between passes)."""
    if not 0 <= start < stop <= blocks or times < 1:
        raise ValueError(f"a loop over blocks {start} .. {stop - 1}, {times} times, does not fit {blocks} blocks")
    plan = [PlanEntry(i) for i in range(start)]
    for t in range(times):
        plan += [PlanEntry(i, inject=Inject(t, t > 0) if inject and i == start else None) for i in range(start, stop)]
    return plan + [PlanEntry(i) for i in range(stop, blocks)]


def _tensors(delta):
    """The tensors of what a block leaves to be added, where it is one of these; else None."""
    if isinstance(delta, torch.Tensor):
        return (delta,)
    if type(delta) is PartialSums:
        return (delta.sums,)
    if type(delta) is Prenormed:
        return delta.xw, delta.sums
    return None


class DecoderLM:
    def __init__(
        self,
        config,
        embedding: Embedding,
        blocks: Sequence[Block],
        plan: Sequence[PlanEntry],
        final_norm: Norm,
        head: Linear,
        tied_head: bool,
        logit_scale: float = 1.0,
        logit_softcap: Optional[float] = None,
        pass_vectors: Optional[PassVectors] = None,
    ):
        """`logit_scale`: the head's result is multiplied by it (in 32-bit).  `logit_softcap`: the
        logits then pass through cap * tanh(logits / cap) (in 32-bit; None: not).
        `pass_vectors`: the vectors that plan entries' `inject` names."""
        self.pass_vectors = pass_vectors
        self.logit_scale = float(logit_scale)
        self.logit_softcap = float(logit_softcap) if logit_softcap else None
        self.config = config
        self.embedding = embedding
        self.blocks = list(blocks)
        self.plan = [
            dataclasses.replace(e, cache=i if e.cache is None else e.cache) for i, e in enumerate(plan)
        ]
        self.final_norm = final_norm
        self.head = head
        self.tied_head = tied_head
        writers = {e.cache for e in self.plan if e.writes}
        for e in self.plan:
            if not 0 <= e.block < len(self.blocks):
                raise ValueError(f"plan names block {e.block}, the model has {len(self.blocks)}")
            if not e.writes and e.cache not in writers:
                raise ValueError(f"plan entry reads cache {e.cache} that no entry writes")
            if e.inject is not None and e.inject.vector is not None:
                if pass_vectors is None or not 0 <= e.inject.vector < pass_vectors.count:
                    raise ValueError(f"plan entry adds pass vector {e.inject.vector}, which the model does not have")

    # -- structure ---------------------------------------------------------
    @property
    def vocab_size(self) -> int:
        return self.embedding.vocab_size

    @property
    def max_positions(self) -> Optional[int]:
        """Most tokens of one request, where the model has a bound of its own (a table of position vectors)."""
        return getattr(self.embedding, "max_positions", None)

    def tensor_specs(self) -> Dict[str, TensorSpec]:
        specs: Dict[str, TensorSpec] = dict(self.embedding.tensor_specs())
        for b in self.blocks:
            specs.update(b.tensor_specs())
        if self.pass_vectors is not None:
            specs.update(self.pass_vectors.tensor_specs())
        specs.update(self.final_norm.tensor_specs())
        specs.update(self.head.tensor_specs())
        return specs

    def cache_layers(self):
        """cache id -> the mixer that defines its needs (the writer)."""
        out = {}
        for e in self.plan:
            if e.writes:
                mixer = self.blocks[e.block].mixer
                if e.cache in out and out[e.cache] is not mixer:
                    raise ValueError(f"two different mixers write cache {e.cache}")
                out[e.cache] = mixer
        return out

    # -- weights -------------------------------------------------------------
    def bind(self, weights: Dict[str, torch.Tensor], ctx: BuildContext) -> None:
        self.ctx = ctx
        self.embedding.bind(weights, ctx)
        for b in self.blocks:
            b.bind(weights, ctx)
        if self.pass_vectors is not None:
            self.pass_vectors.bind(weights, ctx)
        self.final_norm.bind(weights, ctx)
        head_name = self.head.names[0]
        if head_name in weights:
            self.head.bind(weights, ctx)
        elif self.tied_head:
            self.head.bind_tensor(self.embedding.weight, ctx)
        else:
            raise KeyError(head_name)

    # -- one step --------------------------------------------------------------
    def _injected(self, inject: Inject, delta, step) -> Injected:
        """What the block before has left to be added and what enters the stream ahead of the next block."""
        if isinstance(delta, Carried):  # the block before has added everything into the stream itself
            delta = None
        return Injected(delta, None if inject.vector is None else self.pass_vectors.row(inject.vector),
                        self.embedding.again(step) if inject.embedding else None, self.ctx.ops)

    def _run_layer(self, i: int, hidden, delta, step, caches):
        """Plan entry i: what the block leaves to be added."""
        e, last = self.plan[i], len(self.plan) - 1
        # the norm that the next block starts with, if the products around it may do its work
        if i < last and self.plan[i + 1].inject is not None:
            next_norm = None  # something enters the stream first
        elif i < last:
            follower = self.blocks[self.plan[i + 1].block]
            next_norm = follower.entry_norm()
            if next_norm is None and self.blocks[e.block].chained_norm() is not None:
                next_norm = follower.chained_norm()  # (between two blocks that chain their norms)
        else:  # the final norm, where the head's product can take its place (every row goes to the head) ...
            next_norm = self.final_norm if step.every_row_wanted and not self.head.has_bias else None
            # ... but not in float32, whose rows' sums do not follow what else the step brings: folded, they run in another order
            if self.ctx.dtype == torch.float32 and self.blocks[e.block].chained_norm() is None:
                next_norm = None
        if e.inject is not None:
            delta = self._injected(e.inject, delta, step)
        return self.blocks[e.block].forward(hidden, delta, step, caches.layer(i), next_norm=next_norm)

    # Layers that are alike (csrc/record.py): worth it from two layers launched again on, the host's checks of all layers being about a
    # layer's launches again (28 layers: 0.2 ms).  Steps of more tokens keep the device busy for longer than the host needs, and what a layer made would
    # be held for longer than before.
    ALIKE_LAYERS, ALIKE_TOKENS = 6, 2048

    def _alike_layers(self, step, caches):
        """(first entry to record, end, [(operands, their addresses)] of the entries from the first on): the entries first - 1 ..
        end - 1 have blocks that launch alike; None without such a stretch."""
        ops, plan = self.ctx.ops, self.plan
        if (len(plan) < self.ALIKE_LAYERS or step.token_ids.shape[0] > self.ALIKE_TOKENS
                or not getattr(ops, "may_record", lambda: False)() or not parts_as_written()):
            return None
        best, start, seen, settings, kinds, like = None, 0, [], None, None, None  # the stretch: first entry, (tensors, addresses), what its blocks share
        for i, e in enumerate(plan):
            made = self.blocks[e.block].launches() if e.inject is None else None
            cache = caches.layer(i)
            if made is None or cache.kv is None or cache.state is not None:
                settings = None
                continue
            tensors = made[1] + (cache.kv,)
            if settings is not None and made[0] == settings and cache.group is like.group and cache.writes == like.writes:
                at = addresses_of(tensors, kinds)
                if at is not None:
                    seen.append((tensors, at))
                    continue
            start, settings, like, kinds = i, made[0], cache, operand_kinds(tensors)
            seen = [(tensors, addresses_of(tensors, kinds))]
            if seen[0][1] is None:
                settings = None
            elif best is None or len(best[1]) < self.ALIKE_LAYERS:
                best = (start, seen)
        if best is None or len(best[1]) < self.ALIKE_LAYERS:
            return None
        start, seen = best
        # the last product of a layer may do the work of the norm that its follower starts with
        out = []
        for k in range(1, len(seen) - 1):
            w = self.blocks[plan[start + k + 1].block].input_norm().weight
            out.append((seen[k][0] + (w,), seen[k][1] + [w.data_ptr()]))
        return start + 1, start + len(seen), out

    def _run_alike(self, stretch, hidden, delta, step, caches):
        """The recorded entry and those behind it but for the stretch's last, whose follower is another: (what the last of them
        leaves, the entry that comes next)."""
        first, end, operands = stretch
        ops, given = self.ctx.ops, _tensors(delta)
        record = ops.record()
        try:
            left = self._run_layer(first, hidden, delta, step, caches)
        finally:
            ops.end_record()
        if given is None or type(left) is not type(delta) or getattr(left, "eps", None) != getattr(delta, "eps", None):
            return left, first + 1
        replay = Replay(record, operands[0][0], given, _tensors(left))
        if not replay.ok:
            return left, first + 1
        with torch.no_grad():  # (a product into a tensor that is there has no gradient, whatever its weight asks for)
            for tensors, addresses in operands[1:]:
                ops.replay(replay, tensors, addresses)
        return left, end - 1

    def forward(self, step, caches) -> torch.Tensor:
        """Run the tokens of `step` (engine.batch.StepState) through the plan and
        return float32 logits [len(step.logit_rows), vocab]."""
        step.scratch.clear()  # per-step tables are made anew in every run (also when a graph is captured)
        first_norm = None
        if self.plan and self.plan[0].inject is None:  # (nothing enters the stream between the embedding and the norm)
            first_norm = self.blocks[self.plan[0].block].input_norm()
        if first_norm is not None:
            hidden, delta = self.embedding.forward(step.token_ids, step, norm=first_norm)
        else:
            hidden, delta = self.embedding.forward(step.token_ids, step), None
        stretch = self._alike_layers(step, caches)
        i = 0
        while i < len(self.plan):
            if stretch is not None and i == stretch[0]:
                delta, i = self._run_alike(stretch, hidden, delta, step, caches)
            else:
                delta, i = self._run_layer(i, hidden, delta, step, caches), i + 1
        if step.logit_rows.shape[0] == 0:
            return torch.empty((0, self.vocab_size), dtype=torch.float32, device=hidden.device)
        if isinstance(delta, Carried):  # the last block has added everything into the stream itself
            delta = None
        if isinstance(delta, Normed):  # the final norm of every row, made by the last block's last launch
            x = delta.x
        else:
            x = delta if isinstance(delta, Prenormed) else self.final_norm.forward(hidden, delta, rows=step.logit_rows)
        logits = self.head.forward(x, out_dtype=torch.float32)
        if self.logit_scale != 1.0:
            logits = self.ctx.ops.scale_(logits, self.logit_scale)
        return logits if self.logit_softcap is None else self.ctx.ops.softcap_(logits, self.logit_softcap)
