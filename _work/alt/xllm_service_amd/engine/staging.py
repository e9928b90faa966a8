"""One host-to-device copy for all the small arrays of a step.

A copy costs the host 10 us from pinned memory and 20-40 us from pageable
memory (which also waits for the stream to drain), whatever its size here; a
step has five to nine such arrays. Sections start at multiples of 16 bytes.
"""
from __future__ import annotations

from typing import List, Sequence, Tuple

import numpy as np
import torch

WORD = 4                 # sections are counted in 32-bit words


def _words(shape, dtype) -> int:
    return int(np.prod(shape, dtype=np.int64)) * np.dtype(dtype).itemsize // WORD


def _layout(parts) -> Tuple[List[int], List[int], int]:
    """(sizes, starts, total) in words of (shape, dtype) sections."""
    sizes = [_words(s, d) for s, d in parts]
    starts, at = [], 0
    for n in sizes:
        starts.append(at)
        at += -(-n // 4) * 4
    return sizes, starts, at


def _torch_view(t: torch.Tensor, shape, dtype) -> torch.Tensor:
    if dtype == np.int64:
        t = t.view(torch.int64)
    return t if len(shape) == 1 else t.view(shape)


def upload(arrays: Sequence[np.ndarray], device) -> List[torch.Tensor]:
    """The int32 and int64 arrays as tensors on the device, from one copy. On a GPU
    it is asynchronous: the pinned block returns to torch's host allocator, which
    keeps it until the stream has passed the copy."""
    parts = [(a.shape, a.dtype) for a in arrays]
    sizes, _, total = _layout(parts)
    cuda = torch.device(device).type == "cuda"
    flat = torch.empty(total, dtype=torch.int32, pin_memory=cuda)
    host, at, cuts = flat.numpy(), 0, []
    for a, n in zip(arrays, sizes):
        host[at:at + n] = np.ascontiguousarray(a).reshape(-1).view(np.int32)
        pad = -n % 4
        host[at + n:at + n + pad] = 0
        at += n + pad
        cuts += [n, pad]
    pieces = flat.to(device, non_blocking=cuda).split(cuts)
    return [_torch_view(t, *p) for t, p in zip(pieces[::2], parts)]


class Staging:
    """Device buffers of a captured graph, all in one block, and their pinned
    image: `host[name]` (numpy) is filled, then flush() copies the block, or its
    part up to `rows` rows of the last section."""

    def __init__(self, sections, device):
        # (name, shape, numpy type, fill)
        parts = [(s, np.dtype(d)) for _, s, d, _ in sections]
        sizes, starts, total = _layout(parts)
        self._pin = torch.zeros(total, dtype=torch.int32,
                                pin_memory=torch.device(device).type == "cuda")
        host = self._pin.numpy()
        self.host = {}
        for (name, shape, dtype, fill), n, at in zip(sections, sizes, starts):
            self.host[name] = host[at:at + n].view(dtype).reshape(shape)
            self.host[name][...] = fill
        self._dev = self._pin.to(device, copy=True)
        self.dev = {name: _torch_view(self._dev[at:at + n], *p) for
                    (name, *_), n, at, p in zip(sections, sizes, starts, parts)}
        self._last = starts[-1]
        self._row = _words(parts[-1][0][1:], parts[-1][1])
        self._copied = None

    def wait(self) -> None:
        """Block until the copy of the previous replay has read the pinned image;
        only then may the host refill it. A caller that syncs every step (sampling
        does) never waits here, one that replays without reading results back would
        otherwise race."""
        if self._copied is not None:
            self._copied.synchronize()

    def flush(self, rows: int) -> None:
        n = self._last + rows * self._row
        self._dev[:n].copy_(self._pin[:n], non_blocking=True)
        if not self._dev.is_cuda:
            return
        if self._copied is None:
            self._copied = torch.cuda.Event()
        self._copied.record()
