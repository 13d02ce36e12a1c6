"""A step of few single tokens, or of short prompts, through all layers in one launch (``csrc/chain.hip``, ``chain_prompt.hip``).

A part that the launch takes says what of it there is (``chain_link``); a model whose every layer does, over one cache and one
rotation, runs such steps through it, and all others -- other mixers, options, types, sizes, more rows, longer sequences --
through the layers' own kernels."""

from __future__ import annotations

import threading
from contextlib import contextmanager
from typing import Dict, List, Optional

import torch

_turn = threading.RLock()
_last: Dict[int, torch.cuda.Stream] = {}  # by GPU: the stream of the last launch of all layers


@contextmanager
def in_turn(device: torch.device, launches: bool = True):
    """Around a launch of all layers, or a replay that holds one: puts it behind the one before it on this GPU, whatever streams and
    threads the two come from.  Two at once could each fill a die for the other, whose blocks then wait until they give up
    (``csrc/chain.h``).  One stream's follow one another by themselves; inside a capture nothing runs."""
    if not launches or torch.cuda.is_current_stream_capturing():
        yield
        return
    with _turn:
        stream = torch.cuda.current_stream(device)
        last = _last.get(device.index)
        if last is not None and last != stream:
            stream.wait_stream(last)
        _last[device.index] = stream
        yield


@contextmanager
def turns_waited_for(device: torch.device):
    """Around launches at whose end the caller waits for the whole GPU: nobody has to get behind them afterwards."""
    with _turn:
        yield
        _last.pop(device.index, None)


class LayerChain:
    def __init__(self, links: List[dict], rt):
        """``links``: what each run of the schedule says of itself (``PreNormBlock.chain_link``)."""
        self.links, self.device = links, rt.device
        first = links[0]
        self.sizes = {name: first[name] for name in ("width", "heads", "kv_heads", "head_dim", "inner")}
        self.sizes["dtype"] = rt.dtype
        self.eps, self.scale, self.position, self.gain_dtype = first["eps"], first["scale"], first["position"], first["gains"][0].dtype
        # where a wait that was given up says so: a word of host memory that the kernel writes
        self.failed = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        self._failed = self.failed.numpy()
        self._lost = 0
        self.tables: Dict[tuple, torch.Tensor] = {}  # the layers' pointers -> the same on the device
        self.exchange: Optional[torch.Tensor] = None  # where a launch's blocks hand on their words; what lies there between launches is nothing

    @classmethod
    def of(cls, schedule_layers, rt) -> Optional["LayerChain"]:
        links = []
        for layer in schedule_layers:
            link = layer.chain_link(rt) if hasattr(layer, "chain_link") else None
            if link is None:
                return None
            links.append(link)
        alike = ("width", "heads", "kv_heads", "head_dim", "inner", "eps", "scale", "position")
        if not links or any(link[name] != links[0][name] for link in links for name in alike):
            return None
        if any(gain.dtype != links[0]["gains"][0].dtype or gain.data_ptr() % 16 for link in links for gain in link["gains"]):
            return None
        if rt.is_fp32 and any(t.dtype != torch.float32 or not t.is_contiguous() or t.data_ptr() % 16
                              for link in links for t in (*link["weights"], *link["gains"])):
            return None
        chain = cls(links, rt)
        return chain if rt.ops.chain_takes(len(links), 1, **chain.sizes) else None

    def plan(self, batch: int, longest: int, rt):
        """(runs of a sequence's keys, waves of a run) for a step of these sizes, or None: the layers' own kernels."""
        return rt.ops.chain_plan(len(self.links), batch, longest, **self.sizes)

    def takes_prompt(self, rows: int, rt) -> bool:
        """Whether the launch takes a step of prompts of this many rows in all that each begin at their sequence's first position."""
        return rt.ops.chain_prompt_takes(len(self.links), rows, **self.sizes)

    def lost(self) -> int:
        """How often a report of given-up waits has been found: one more than before if a step that has run since then made one.
        (Steps still on their way may make another for the same reason: they are waited for, and go with it.)"""
        if self._failed[0]:
            torch.cuda.current_stream().synchronize()
            self._failed[0] = 0
            self._lost += 1
        return self._lost

    def views_fit(self, views) -> bool:
        """Whether each layer writes keys and values of its own, through one block table."""
        return all(not getattr(view, "read_only", True) and view.k_pages.dtype == self.sizes["dtype"]
                   and view.block_table.data_ptr() == views[0].block_table.data_ptr() for view in views)

    def _table(self, views, device) -> Optional[torch.Tensor]:
        key = tuple(pointer for link, view in zip(self.links, views)
                    for pointer in (*(w.data_ptr() for w in link["weights"]), *(g.data_ptr() for g in link["gains"]),
                                    view.k_pages.data_ptr(), view.v_pages.data_ptr()))
        table = self.tables.get(key)
        if table is None:
            if torch.cuda.is_current_stream_capturing():
                return None  # (the copy below does not belong into a graph; a graph's eager run comes first)
            while len(self.tables) >= 16:
                self.tables.pop(next(iter(self.tables)))  # (graphs hold what they were captured with: ``held``)
            table = self.tables[key] = torch.tensor(key, dtype=torch.int64).to(device)
        return table

    def _room(self, words: int) -> Optional[torch.Tensor]:
        """The exchange, of ``words`` 32-bit words at least: one for all launches, as they follow one another (``in_turn``).  It grows by powers of two, and not
        inside a capture (None; a graph's eager run comes first, and a graph holds the one that it was captured with: ``held``)."""
        if self.exchange is None or self.exchange.numel() < words:
            if torch.cuda.is_current_stream_capturing():
                return None
            self.exchange = torch.empty(1 << (words - 1).bit_length(), dtype=torch.int32, device=self.device)
            self._exchange_of = torch.cuda.current_stream()
        elif not torch.cuda.is_current_stream_capturing() and torch.cuda.current_stream() != self._exchange_of:
            self.exchange.record_stream(torch.cuda.current_stream())  # (it may be let go while that stream's launch runs)
        return self.exchange

    def held(self) -> List[torch.Tensor]:
        """What a captured launch has the addresses of."""
        return [*self.tables.values(), *([self.exchange] if self.exchange is not None else [])]

    def forward(self, x: torch.Tensor, ctx, views, plan, rt):
        """The stream, and what the last layer still adds to it; None where the launch cannot be made here."""
        table = self._table(views, x.device)
        if table is None:
            return None
        tables = ctx.step_tables(rt, self.position.rotary(), views[0].block_table)
        more = dict(self.sizes, room=self._room, gain_dtype=self.gain_dtype, eps=self.eps, scale=self.scale)
        with in_turn(self.device):
            if plan == "prompt":
                done = rt.ops.chain_prompt(table, len(self.links), x, tables, ctx.tok_pos, self.failed, **more)
            else:
                done = rt.ops.chain(table, len(self.links), x, tables, ctx.tok_pos, plan, self.failed, **more)
        ctx.chained = done is not None
        return done
