"""An activation that is the norm of the residual stream, not yet computed.

A block hands ``Normed(x, norm)`` to a mixer or feed-forward that declares
``accepts_lazy_norm``; :func:`parts.linear.linear` then fuses the norm into the
product where a kernel can -- or takes what the product before has prepared for
this norm (``pre``) -- and otherwise calls :meth:`tensor`, which runs the norm
once and keeps the result.
"""
from __future__ import annotations

from typing import Any, Dict, Optional, Tuple

import torch

from ..errors import EngineError


class Normed:
    def __init__(self, x: torch.Tensor, norm, ctx=None, rows: Optional[torch.Tensor] = None,
                 n_rows: Optional[int] = None, pre=None, done: Optional[torch.Tensor] = None):
        self.x, self.norm, self.ctx, self.rows = x, norm, ctx, rows
        # what the product that last added into x left for this norm (ops.Prenormed), if anything
        self.pre = pre if rows is None else None
        self.n_rows = x.shape[0] if rows is None and n_rows is None else (n_rows if n_rows is not None else rows.numel())
        self._tensor: Optional[torch.Tensor] = done      # (``done``: the product before has computed the norm already)

    def tensor(self) -> torch.Tensor:
        if self._tensor is None:
            self._tensor = self.norm.forward(self.x, self.ctx, rows=self.rows, n_rows=self.n_rows if self.rows is not None else None)
        return self._tensor

    def fusable_scale(self):
        """(scale vector, eps) if the norm is a plain RMSNorm that a product may absorb, else None."""
        f = getattr(self.norm, "fusable", None)
        return f() if f is not None else None


class _Reading:
    """While it is entered, the handoff's reading_next is what it was given (NormHandoff.reader)."""

    def __init__(self, handoff: "NormHandoff", reading: Optional[Tuple[Any, bool]]):
        self.handoff, self.reading, self.before = handoff, reading, None

    def __enter__(self) -> None:
        self.before, self.handoff.reading_next = self.handoff.reading_next, self.reading

    def __exit__(self, *exc) -> None:
        self.handoff.reading_next = self.before


class NormHandoff:
    """The whole protocol by which a product that adds into the residual stream prepares the norm that reads the
    stream next, in one place (a step's StepContext carries one).  Three parties use it:

    the model    ``begin_entry(layer, following, n_rows)`` before every schedule entry: what the entry before left
                 for this entry's first norm stays, everything else goes, and the first reader of the entry after
                 this one is noted (``first_reader(n_rows) -> (norm, takes_parts)`` of a block that has one);
                 ``begin_step()`` before the first and ``end_step()`` after the last.
    a block      ``with handoff.reader(norm, takes_parts):`` around each part that adds into the stream, naming the
                 norm that reads the stream after that part (``handoff.next_entry`` for its last part), and
                 ``take(norm)`` for what was left for a norm of its own.
    a product    (parts.linear.linear) ``reading_next`` -- (norm, takes_parts) or None -- and ``leave(norm, what)``.

    What is left is the finished norm (ops.Finished), which serves every reader, or -- only for a reader that says
    it takes them -- the parts of one that a product can finish (ops.Prenormed).  Nothing left outlives the entry
    after the one that made it.  A block that does not use any of this stays correct: its norms simply run.

    ``owe(reader, what)`` leaves something of another kind, which the stream lacks until the reader has added it (a
    sublayer's output for parts.block.AddingReader).  Only a block that takes it in its own forward names such a reader; the
    entry after this one has to, and where it does not the step ends in an error instead of without that output."""

    def __init__(self):
        self.reading_next: Optional[Tuple[Any, bool]] = None
        self.next_entry: Optional[Tuple[Any, bool]] = None
        self._left: Dict[int, Any] = {}
        self._owed: Optional[Tuple[Any, Any]] = None       # (reader, what) of the entry that runs
        self._due = False                                  # ... and it was owed to that entry when it began

    @staticmethod
    def _first_reader(layer, n_rows: int) -> Optional[Tuple[Any, bool]]:
        first = getattr(layer, "first_reader", None)
        return first(n_rows) if first is not None else None

    def begin_step(self) -> None:
        self._left.clear()
        self.next_entry = self.reading_next = self._owed = None

    def begin_entry(self, layer, following, n_rows: int) -> None:
        mine = self._first_reader(layer, n_rows)
        if self._owed is not None and (self._due or mine is None or mine[0] is not self._owed[0]):
            self._fail()
        self._due = self._owed is not None
        kept = self._left.pop(id(mine[0]), None) if mine is not None else None
        self._left.clear()
        if kept is not None:
            self._left[id(mine[0])] = kept
        self.next_entry = self._first_reader(following, n_rows) if following is not None else None
        self.reading_next = None

    def end_step(self) -> None:
        if self._owed is not None:
            self._fail()
        self.begin_step()

    def _fail(self) -> None:
        reader = self._owed[0]
        self.begin_step()
        raise EngineError(f"a layer's output was left to {type(reader).__name__}, which did not add it to the stream")

    def reader(self, norm, takes_parts: bool = False) -> "_Reading":
        return _Reading(self, (norm, bool(takes_parts)) if norm is not None else None)

    def leave(self, norm, what) -> None:
        self._left[id(norm)] = what

    def owe(self, reader, what) -> None:
        if self._owed is not None:
            self._fail()
        self._owed, self._due = (reader, what), False

    def take(self, norm):
        if self._owed is not None and self._owed[0] is norm:
            owed, self._owed = self._owed[1], None
            return owed
        return self._left.pop(id(norm), None)
