"""Device workspaces that outlive a call, for kernels that hand data from one launch to the next.

Two calls may share a buffer only if the GPU runs them one after the other, so each stream has
its own, and the graphs captured on a device share one that no eager call uses: replays of
different graphs (and the branches of one) must be ordered among themselves, as one stream
orders them, but need no order against eager calls.
"""

from __future__ import annotations

import torch

# Outgrown buffers that a captured graph still launches on.  They are never freed: their memory
# would be handed to new tensors.  Growth at least doubles, so they add up to less than what
# replaced them.
retired: list[torch.Tensor] = []

# Streams besides the default one that keep a buffer, per device and kind of workspace; beyond
# it the oldest is freed (in the order of its own stream, where the allocator reuses it).
_SIDE_STREAMS = 64


class Workspaces:
    """The buffers of one kind of workspace, by device and stream."""

    def __init__(self, what: str, reserve: str):
        self.what, self.reserve = what, reserve
        self.default: dict[int, torch.Tensor] = {}  # by device: the default stream's
        self.side: dict[tuple[int, int], torch.Tensor] = {}  # by device and stream handle
        self.captured: dict[int, torch.Tensor] = {}  # by device: the captured graphs'

    def ready(self, index: int, stream: int, nbytes: int) -> torch.Tensor | None:
        """The buffer of an eager call on the default stream, if it is there and large enough: what
        nearly every call finds.  get() alone made host-bound calls 0.6 us slower (14.9 -> 15.6)."""
        if stream == 0:
            ws = self.default.get(index)
            if ws is not None and ws.numel() >= nbytes and ws is not self.captured.get(index):
                return ws
        return None

    def get(self, device: torch.device | str | int, nbytes: int, least: int | None = None,
            optional: bool = False) -> torch.Tensor | None:
        """At least `nbytes` for calls on the device's current stream.  Inside a capture nothing
        is allocated: the largest buffer that the device has becomes the graphs' if it holds
        `nbytes`, or `least` at least, and the eager calls that used it get another.  Without
        such a buffer the capture fails, or gets None where the workspace is `optional`."""
        dev = torch.device(device) if not isinstance(device, int) else torch.device("cuda", device)
        i = dev.index if dev.index is not None else torch.cuda.current_device()
        stream = torch._C._cuda_getCurrentRawStream(i)
        if stream == 0:
            ws = self.default.get(i)
            mine = ws is not self.captured.get(i)
        elif torch.cuda.is_current_stream_capturing():
            return self._for_capture(i, nbytes, nbytes if least is None else least, optional)
        else:
            ws = self.side.get((i, stream))
            mine = True
        if ws is None or ws.numel() < nbytes or not mine:
            size = max(nbytes, 256)
            if ws is not None:
                size = max(size, ws.numel() if ws.numel() >= nbytes else 2 * ws.numel())
            # An outgrown buffer is freed here: only calls on this stream used it.
            ws = torch.empty(size, dtype=torch.uint8, device=torch.device("cuda", i))
            if stream == 0:
                self.default[i] = ws
            else:
                self.side[i, stream] = ws
                for old in [k for k in list(self.side) if k[0] == i][:-_SIDE_STREAMS]:
                    self.side.pop(old, None)
        return ws

    def _for_capture(self, i: int, nbytes: int, least: int, optional: bool) -> torch.Tensor | None:
        own = self.captured.get(i)
        if own is not None and own.numel() >= nbytes:
            return own
        spare = [(None, self.default[i])] if i in self.default and self.default[i] is not own else []
        spare += [(k, ws) for k, ws in list(self.side.items()) if k[0] == i]
        key, best = max(spare, key=lambda kw: kw[1].numel(), default=(None, None))
        if best is not None and best.numel() >= (nbytes if own is not None and own.numel() >= least else least):
            if own is not None:
                retired.append(own)
            if key is not None:
                self.side.pop(key, None)
            self.captured[i] = best
            return best
        if own is not None and own.numel() >= least:
            return own
        if optional:
            return None
        raise RuntimeError(f"the {self.what} workspace must be reserved before graph capture "
                           f"({nbytes} bytes needed): call {self.reserve}() first")
