"""Drawing one token per sequence from float32 logits on the GPU.

The draw of sequence s at its step t uses the uniform number that
Philox4x32-10 gives for key = seed and counter = (t, s, 0, 0): it does not
depend on which other sequences share the batch."""
from __future__ import annotations

import time
from typing import List, Sequence

import torch

from ..kernels import ops
from .config import SamplingConfig


LOOK_FOR = 1e-4       # seconds that the host looks at the memory of tokens that it wants at once (`Sampler.sample`) before it waits for the
                      # draw's event instead: an event behind a kernel is known 9 us after it, a token that the kernel wrote at once (16 rows
                      # of 131,072: 49 and 42 us a draw).  Looking keeps the interpreter, so a draw with a step behind it is only waited for


class _Place:
    """Pinned host memory of one draw: what its kernel reads, the (sequence, step) pairs, and writes, the tokens.  The kernel goes by
    their addresses, of which torch's allocator knows nothing, so the memory is held until the draw is over."""
    done = None                          # the event behind the draw that uses it, None once that is known to be over

    def __init__(self, cap: int):
        self.counters = torch.empty((cap, 2), dtype=torch.int32, pin_memory=True)
        self.tokens = torch.empty((cap,), dtype=torch.int32, pin_memory=True)
        self.pairs, self.ids = self.counters.numpy(), self.tokens.numpy()

    def wait(self) -> None:
        if self.done is not None:
            self.done.synchronize()
            self.done = None

    def __del__(self):
        self.wait()


class Drawn:
    """The tokens of one draw: on the device at once (`device`, int32 [B], valid until the
    sampler's next draw has been launched), on the host when `tokens()` is asked for (until two
    more draws have been launched)."""

    def __init__(self, device: torch.Tensor, place: _Place):
        self.device, self._place, self._done, self._tokens = device, place, place.done, None

    def tokens(self) -> List[int]:
        if self._tokens is None:
            self._done.synchronize()
            self._take()
        return self._tokens

    def _take(self) -> None:
        if self._place.done is self._done:
            self._place.done = None
        self._tokens = self._place.ids[:self.device.shape[0]].tolist()

    def tokens_at_once(self) -> List[int]:
        """`tokens()` for a caller that has nothing else to do meanwhile.  What the draw leaves on the device is there for the draw's
        own stream only when this returns."""
        if self._tokens is None:
            ids = self._place.ids[:self.device.shape[0]]
            # a row's token, never negative, is the last that its workgroup does with the memory: where all are there it may be used again
            until = time.perf_counter() + LOOK_FOR
            while ids.size and ids.min() < 0:
                if time.perf_counter() > until:
                    return self.tokens()
            self._take()
        return self._tokens


class Sampler:
    def __init__(self, config: SamplingConfig, device):
        self.config = config
        self.device = device
        self._probs = None
        self._lists = None               # the lists of rows in parts, of the last draw's shape and options
        self._lists_for = None           # (the options may change between draws, and with them whether rows go in parts)
        self._out = None
        self._places = None              # two, used in turn: a draw may be launched while the one before is read
        self._turn = 0
        self._last = None                # the event behind the last draw

    def draw(self, logits: torch.Tensor, seq_ids: Sequence[int], steps: Sequence[int]) -> Drawn:
        """logits: float32 [B, V] on the GPU -> B token ids, without waiting for them: the
        kernel is launched, which takes the pairs from pinned memory and leaves the tokens there, `Drawn.tokens()` waits."""
        B, V = logits.shape
        c = self.config
        if self._out is None or self._out.shape[0] < B:
            cap = max(B, 64)
            self._places = [_Place(cap) for _ in range(2)]
            self._out = torch.empty((cap,), dtype=torch.int32, device=logits.device)
        if self._probs is None or self._probs.shape[0] < B or self._probs.shape[1] != V:
            self._probs = torch.empty((B, V), dtype=torch.float32, device=logits.device)
        wanted = (B, V, float(c.temperature), int(c.top_k or 0))
        if self._lists_for != wanted:
            self._lists = ops.sample_lists(*wanted, logits.device)
            self._lists_for = wanted
        place = self._places[self._turn]
        self._turn ^= 1
        place.wait()                                 # the memory is free to be written again
        place.pairs[:B, 0] = seq_ids
        place.pairs[:B, 1] = steps
        place.ids[:B] = -1
        ops.sample_kept(logits.contiguous(), wanted[2], wanted[3], float(c.top_p or 0.0), int(c.seed), place.counters, self._probs, self._out,
                        self._lists, place.tokens)
        self._last = place.done = torch.cuda.Event()
        place.done.record()
        return Drawn(self._out[:B], place)

    def sample(self, logits: torch.Tensor, seq_ids: Sequence[int], steps: Sequence[int]) -> List[int]:
        """logits: float32 [B, V] on the GPU -> B token ids."""
        return self.draw(logits, seq_ids, steps).tokens_at_once()

    def last_distribution(self, B: int) -> torch.Tensor:
        """The probabilities the last draw was made from (temperature > 0), there for any stream."""
        self._last.synchronize()
        return self._probs[:B]
