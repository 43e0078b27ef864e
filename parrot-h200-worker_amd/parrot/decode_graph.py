"""HIP-graph replay of cached decode steps.

A decode step of the HIP backend has static shapes: the attention kernels
read the generation position from ``GenerationState.position_device`` and the
step advances it on the device.  ``DecodeGraph`` captures one
``Parrot.decode_step`` for a given state once and replays it per token, which
removes the host launch cost of the ~30 kernels per layer (the reference
reaches the same end on Apple GPUs with fused decode kernels,
parrot/metal_moe.py:182-221 and parrot/model.py:832-925).
"""
from __future__ import annotations

import bisect

import torch
from torch import Tensor

from . import hip_moe
from .model import GenerationState, LocalKVCache, Parrot


def split_forms(start: int, limit: int, line: int | None) -> list[tuple[bool, int]]:
    """The forms of the step (whether every layer that ever splits its keys does)
    that a generation from position ``start`` to ``limit`` comes to, each with
    the position whose step is captured.  ``line``: the first position of the
    split form, or None."""
    if line is None or line >= limit:
        return [(False, start)]
    if start >= line:
        return [(True, start)]
    return [(False, start), (True, limit - 1)]


class DecodeGraph:
    """Captured ``decode_step`` for one generation state.

    ``step(ids)`` appends one token per sequence (ids ``[batch, 1]``) and
    returns the next greedy tokens ``[batch, 1]`` (or the logits
    ``[batch, 1, vocab]`` with ``logits=True``), exactly as
    ``model.decode_next`` / ``model.decode_step`` would on the same state.
    The returned tensor is the graph's static output, overwritten by the next
    step; for greedy tokens it is the graph's input buffer itself (the step's
    last launch writes the tokens there), so feeding it back to ``step``
    costs no copy.  Both run in inference mode, as ``prefill`` /
    ``decode_step`` do.  The state must stay with this object: eager decode
    steps on it in between are allowed (they advance both positions
    consistently).
    """

    @torch.inference_mode()
    def __init__(self, model: Parrot, state: GenerationState, logits: bool = False):
        if state.position_device is None:
            raise RuntimeError("DecodeGraph needs a generation state from a HIP-backend prefill")
        if model.training:
            raise RuntimeError("DecodeGraph requires model.eval()")
        self.model, self.state, self.logits = model, state, logits
        device = state.position_device.device
        self.ids = torch.zeros((state.batch_size, 1), dtype=torch.long, device=device)
        start = state.position
        limit = model.config.max_seq_len
        if start >= limit:
            raise ValueError("Generation state has reached max_seq_len")
        # The step's attention splits the keys of long contexts over workgroups
        # (hip_moe.decode_split_bytes), a choice of launches made when a graph is
        # captured: one graph per form that the generation comes to, all captured
        # here, so that no step waits for a capture or fails in one.  Both forms
        # are right at every position.
        self.out: Tensor | None = None
        self.graphs: dict[bool, torch.cuda.CUDAGraph] = {}
        self._line = self._split_line(limit)
        forms = split_forms(start, limit, self._line)
        try:
            # One eager step on a side stream fills every lazily built cache
            # (packed weights, absorbed maps, RoPE tables, scratch buffers);
            # its cache row at `start` is rewritten by the first real step.
            side = torch.cuda.Stream(device)
            side.wait_stream(torch.cuda.current_stream(device))
            try:
                with torch.cuda.stream(side):
                    out = self._run()
            finally:
                torch.cuda.current_stream(device).wait_stream(side)
            self._rewind(start)
            # Every graph writes the same output tensor.
            self.out = torch.empty_like(out) if self.logits else self.ids
            for splits, position in forms:
                # The device position, which the captured launches read, stays
                # what it is: the host's alone chooses the form.
                self.state.position = position
                self._capture(splits)
        finally:  # no step has been taken, also where the eager one or a capture raised
            self._rewind(start)

    def _split_line(self, limit: int) -> int | None:
        """The first position from which on every layer that splits its keys at
        the longest context does; None: no layer ever does."""
        c, b = self.model.config, self.state.batch_size
        shapes = {(c.n_heads, c.n_kv_heads, c.head_dim, cache.key.shape[2], c.window_size)
                  if isinstance(cache, LocalKVCache) else
                  (c.n_heads, 1, c.kv_latent_dim, cache.latent.shape[1], cache.latent.shape[1])
                  for cache in self.state.layers}
        lines = [bisect.bisect_left(range(limit), True, key=lambda p: bool(
            hip_moe.decode_split_bytes(b, *shape, p + 1)))
            for shape in shapes if hip_moe.decode_split_bytes(b, *shape, limit)]
        return max(lines, default=None)

    @property
    def graph(self) -> torch.cuda.CUDAGraph:
        """The captured step that the next ``step`` replays."""
        return self.graphs[self._form()]

    def _form(self) -> bool:
        """The captured form that the step at the state's position takes."""
        splits = self._line is not None and self.state.position >= self._line
        return splits if splits in self.graphs else not splits

    def _capture(self, splits: bool) -> None:
        graph = torch.cuda.CUDAGraph()
        # One pool for all: the graphs never run at the same time.
        pool = next(iter(self.graphs.values())).pool() if self.graphs else None
        with torch.cuda.graph(graph, pool=pool):
            self._run()
        self.graphs[splits] = graph

    def _run(self) -> Tensor:
        if self.logits:
            out, _ = self.model.decode_step(self.ids, self.state, _out=self.out)
        else:
            # The tokens land in the input buffer, read by the next replay's
            # first launch (the embedding gather), after this step's reads.
            out, _ = self.model.decode_step(self.ids, self.state, _next_token_only=True,
                                            _out=self.ids)
        return out

    def _rewind(self, position: int) -> None:
        self.state.position = position
        self.state.position_device.fill_(position)

    @torch.inference_mode()
    def step(self, input_ids: Tensor) -> Tensor:
        if input_ids.shape != self.ids.shape:
            raise ValueError("decode input must be [cached batch, 1]")
        if self.state.position >= self.model.config.max_seq_len:
            raise ValueError("Generation state has reached max_seq_len")
        if input_ids.data_ptr() != self.ids.data_ptr():
            self.ids.copy_(input_ids)
        self.graph.replay()
        self.state.position += 1
        return self.out
