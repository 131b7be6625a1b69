"""Packed ("jagged") token container and the token-merger interface.

Mirrors ``src/interface/token_merger.py:10-21, 102-116`` of the reference:
``JaggedTokens{tokens [1, P, C], weight [P], offset [n_seg + 1]}`` with its suffix operators
(``:23-100``, here one HIP kernel each) and the four methods of ``ITokenMerger``.
"""

from __future__ import annotations

from abc import ABC, abstractmethod
from dataclasses import dataclass
from typing import Any, Callable

import torch

from . import _lib


@dataclass
class JaggedTokens:
    tokens: torch.Tensor      # [1, P, C]
    weight: torch.Tensor      # [P]   source tokens per packed row (1 or the window size)
    offset: torch.Tensor      # [n_seg + 1] int64 segment boundaries

    def apply(self, func: Callable[[torch.Tensor], torch.Tensor]) -> "JaggedTokens":
        return JaggedTokens(tokens=func(self.tokens), weight=self.weight, offset=self.offset)

    def add_suffix(self, suffix: torch.Tensor) -> "JaggedTokens":
        """Appends ``suffix[m]`` (``suffix [M, T, C]``, weight 1) to each of the ``M`` segments
        (reference ``src/interface/token_merger.py:23-58``); one HIP kernel."""
        M = self.offset.shape[0] - 1
        if suffix.shape[0] != M:
            raise ValueError(f"suffix batch dim ({suffix.shape[0]}) must match segment count ({M})")
        _lib.require_gpu_tensor(self.tokens, "tokens")
        C = int(suffix.shape[2])
        if self.tokens.shape[2] != C:
            raise ValueError(f"suffix channels ({C}) must match the tokens' ({self.tokens.shape[2]})")
        return JaggedTokens(*_lib.host().add_suffix(self.tokens, self.weight, self.offset, suffix))

    def split_suffix(self, count: int) -> "tuple[JaggedTokens, torch.Tensor]":
        """Strips the last ``count`` rows of every segment (inverse of ``add_suffix``; reference
        ``src/interface/token_merger.py:60-100``).  Returns ``(stripped, suffix [M, count, C])``."""
        M = self.offset.shape[0] - 1
        T, P = int(count), int(self.tokens.shape[1])
        if P - M * T < 0:
            raise ValueError(f"Cannot strip {T} tokens from each of {M} segments (total tokens = {P})")
        _lib.require_gpu_tensor(self.tokens, "tokens")
        stripped = _lib.host().split_suffix(self.tokens, self.weight, self.offset, T)
        if stripped is None:
            raise ValueError(f"count={T} exceeds the length of at least one segment")
        tokens, weight, offset, suffix = stripped
        return JaggedTokens(tokens, weight, offset), suffix


class ITokenMerger(ABC):
    JaggedTokens = JaggedTokens

    @abstractmethod
    def build_ctx(self, feature: torch.Tensor, confidence: torch.Tensor | None = None) -> Any: ...

    @abstractmethod
    def merge(self, ctx: Any, tokens: torch.Tensor, stub: Any | None = None, *,
              start_index: int | None = None) -> tuple[JaggedTokens, Any]: ...

    @abstractmethod
    def split(self, ctx: Any, stub: Any, tokens: JaggedTokens) -> torch.Tensor: ...

    @abstractmethod
    def build_infer_mask(self, ctx: Any) -> torch.Tensor: ...
