"""The description of one step's batch, as the parts see it.

A step holds *segments*: for each request its next tokens (a portion of a prompt, or one decoded
token), laid out flat one after the other. The reference builds a padded rectangle of whole
prompts or a column of single decode tokens, never both
(core/src/worker/model_worker.rs:266-353 and :427-505); here there is one flat form for all.
"""
from dataclasses import dataclass, field
from typing import Dict, Hashable, List, Optional, Sequence, Tuple

import torch


@dataclass
class StepEntry:
    """One request's part of a step: its next tokens and the places among them whose logits are wanted."""

    request_id: Hashable
    tokens: Sequence[int]
    want: Sequence[int] = ()
    # >= 0: the entry is one token that the host does not know yet, row ``prev_row`` of the tokens that the step
    # before this one sampled (``ModelExecutor.step(..., prev_tokens=...)``); ``tokens`` then holds a placeholder
    prev_row: int = -1


class StepBuffer:
    """A step's metadata on the device: one int32 tensor and where its sections lie. A view of a section costs more than
    a microsecond, and a step that the recorded program runs asks for addresses alone: views are made when a part asks."""

    __slots__ = ("tensor", "base", "offsets")

    def __init__(self, tensor: torch.Tensor, offsets: Dict[str, Tuple[int, int]]):
        self.tensor, self.base, self.offsets = tensor, tensor.data_ptr(), offsets

    def view(self, name: str) -> torch.Tensor:
        at, n = self.offsets[name]
        return self.tensor[at:at + n]

    def address(self, name: str) -> int:
        return self.base + 4 * self.offsets[name][0]


@dataclass
class GroupView:
    """What the runs of one cache group need: where this step's keys go and where each request's pages are."""

    slots: torch.Tensor            # int32 [N]: page * page_size + offset of every token of the step
    block_tables: torch.Tensor     # int32 [S, W]: page of logical block b of segment s (0 where none)
    page_size: int

    @classmethod
    def of_buffer(cls, buffer: StepBuffer, group: int, segments: int, width: int, page_size: int) -> "GroupView":
        """The group's sections of a step's buffer, each a tensor once it is asked for."""
        g = cls.__new__(cls)
        g.__dict__.update(page_size=page_size, _buffer=buffer, _group=group, _shape=(segments, width))
        return g

    def __getattr__(self, name: str):
        buffer = self.__dict__.get("_buffer")
        if buffer is None or name not in ("slots", "block_tables"):
            raise AttributeError(name)
        value = buffer.view("slots%d" % self._group) if name == "slots" else \
            buffer.view("tables%d" % self._group).view(self._shape)
        self.__dict__[name] = value
        return value

    def addresses(self) -> Tuple[int, int, int]:
        """(slots, block tables, blocks a segment's table has)."""
        buffer = self.__dict__.get("_buffer")
        if buffer is not None:
            return buffer.address("slots%d" % self._group), buffer.address("tables%d" % self._group), self._shape[1]
        return self.slots.data_ptr(), self.block_tables.data_ptr(), self.block_tables.shape[1]


# the tensors of a step by name, and the sections of its buffer
_SECTIONS = {"token_ids": "token_ids", "positions": "positions", "seg_of_token": "seg_of", "seg_starts": "seg_starts",
             "seg_first_pos": "seg_first", "state_slots": "state_slots", "logit_rows": "logit_rows"}


@dataclass
class StepContext:
    n_tokens: int
    n_segments: int
    token_ids: torch.Tensor        # int32 [N]
    positions: torch.Tensor        # int32 [N]: position of every token in its request
    seg_of_token: torch.Tensor     # int32 [N]: segment every token belongs to
    seg_starts: torch.Tensor       # int32 [S + 1]: first flat index of every segment, then N
    seg_first_pos: torch.Tensor    # int32 [S]: position of every segment's first token (0 = request begins)
    state_slots: torch.Tensor      # int32 [S]: state slot of every segment's request
    logit_rows: torch.Tensor       # int32 [R]: flat indices whose logits are wanted
    n_logit_rows: int
    groups: List[GroupView]
    # a step of single tokens: its tokens, the longest context first (int32 [N]); a kernel whose work grows with
    # the context starts its workgroups in this order
    longest_first: Optional[torch.Tensor] = None
    # host-side facts, for choosing kernels and for parts that loop over segments
    host_seg_starts: List[int] = field(default_factory=list)
    host_seg_lens: List[int] = field(default_factory=list)
    host_seg_first_pos: List[int] = field(default_factory=list)
    host_state_slots: List[int] = field(default_factory=list)
    request_ids: List[Hashable] = field(default_factory=list)
    max_seg_len: int = 0
    max_context: int = 0           # longest context (tokens in cache after this step) among the segments
    all_single: bool = False       # every segment has exactly one token (a pure decode step)
    aux: dict = field(default_factory=dict)   # what a part derived from this batch and keeps for the next layers
    replayed: bool = False         # the step is captured as a graph: parts must decide nothing from host facts
                                   # that change from step to step (max_context is the model's limit then)

    @classmethod
    def of_buffer(cls, buffer: StepBuffer, longest_first: Optional[torch.Tensor], **facts) -> "StepContext":
        """A step whose tensors are sections of ``buffer``, made when they are asked for; ``facts``: the other fields."""
        ctx = cls.__new__(cls)
        ctx.__dict__.update(facts, longest_first=longest_first, _buffer=buffer)
        return ctx

    def __getattr__(self, name: str):
        section, buffer = _SECTIONS.get(name), self.__dict__.get("_buffer")
        if section is None or buffer is None:
            raise AttributeError(name)
        value = self.__dict__[name] = buffer.view(section)
        return value

    def addresses(self) -> Dict[str, Optional[int]]:
        """Where the arrays that the recorded program reads lie on the device."""
        buffer = self.__dict__.get("_buffer")
        if buffer is not None:
            at = {name: buffer.address(name) for name in ("token_ids", "positions", "seg_of", "logit_rows")}
        else:
            at = {"token_ids": self.token_ids.data_ptr(), "positions": self.positions.data_ptr(),
                  "seg_of": self.seg_of_token.data_ptr(), "logit_rows": self.logit_rows.data_ptr()}
        at["longest_first"] = self.longest_first.data_ptr() if self.longest_first is not None else None
        return at
