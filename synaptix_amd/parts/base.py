"""What every part of a layer has in common.

A part owns the names, shapes and storage of its tensors and the launches that compute it.
It receives its sizes and constants as parameters and its tensor-name prefix as a string; it
does not know which model it is in (the reference produces tensor names the same way, from
the layer: crates/synaptix-models/llm/common/src/model.rs:780).
"""
from __future__ import annotations

from dataclasses import dataclass, field
from typing import Optional

import torch


class Part:
    """Base of norms, position encodings, mixers, feed-forwards and blocks."""

    # True: the part's forward only launches kernels on the current stream (no wait for the device, no shape that
    # depends on device data), finds the step's sequences through the context's device arrays alone (a captured
    # step's `ctx.slots`, `ctx.past` and `ctx.new_counts` are placeholders; a running state is reached with
    # StateLayerView.seq_rows / token_rows) and, apart from such a state, writes the same values when it is run
    # again, so that a step that contains it may be captured into a graph and replayed.  False (the default, for
    # parts from elsewhere): the steps of a model that contains it are launched one by one.
    capturable = False

    def tensor_specs(self) -> dict:
        """name -> TensorSpec of every tensor this part reads from the weight source."""
        return {}

    def load(self, get) -> None:
        """Fetch the tensors; `get(name)` returns the tensor on the device in its kept type."""

    def check(self, dtype) -> None:
        """Raise if no kernel takes this part's sizes in the engine's type `dtype`: asked once when an
        engine is made, so that a size is refused before the first step, not in the middle of it."""


@dataclass(frozen=True)
class KvNeed:
    """A mixer that keeps keys and values of the tokens it has seen: all of them, or a window."""
    kv_heads: int
    head_dim: int
    window: Optional[int] = None      # None: all keys
    v_dim: Optional[int] = None       # size of a value where it differs from the keys' (None: head_dim)
    keep_first: int = 0               # with a window: the first keys of a sequence that stay visible for good
    v_heads: Optional[int] = None     # value heads where several kv heads read the values of one (None: kv_heads)
    # query heads a kv head, where the decode kernel that reads a step's work lists takes them (0: no such kernel reads this cache)
    listed_heads: int = field(default=0, compare=False)


def flat_needs(need) -> tuple:
    """A mixer's need as a tuple of simple needs: a mixer that holds several things (keys and values for one half,
    a running state for the other) returns a tuple, which its cache view then mirrors."""
    if need is None:
        return ()
    return tuple(need) if isinstance(need, (tuple, list)) else (need,)


@dataclass(frozen=True)
class StateNeed:
    """A mixer that keeps a state of fixed size for each sequence, zero when the sequence starts."""
    shape: tuple
    dtype: torch.dtype = torch.float32
