"""Pinned host memory that small tables pass through on their way to the device.

A copy from ordinary host memory makes the host wait until everything launched before it has run: the next step's
launches then reach an idle GPU.  From pinned memory the copy is queued like a launch.  Measured in turn on one machine, milliseconds
without and with (two runs of one side differ by 0.1 to 1.1 %): a request of 32 tokens at 0.6B 16.31 and 16.03, 48 tokens of twelve layers
of the 8B shape 62.8 and 62.4, Dokulix 35.0 and 34.5.
"""
from __future__ import annotations

from typing import Optional

import torch


class Staging:
    """One pinned buffer of 32-bit words, filled again only when its copy has ended: the host is at most one copy ahead of the
    device, whichever streams they went to.  (Four buffers in turn: 16.01 and 16.05, 62.48 and 62.47, 34.48 and 34.51 ms of the above.)

    ``recorded``: under a stream capture.  Nothing is waited for and the copy is recorded as it is: a replay brings what then lies in the buffer."""

    def __init__(self):
        self._buffer: Optional[torch.Tensor] = None
        self._sent: Optional[torch.cuda.Event] = None

    def wait(self) -> None:
        """Waits until the last copy has ended, and with it all that was launched before it on its stream."""
        if self._sent is not None:
            self._sent.synchronize()

    def take(self, words: int, recorded: bool = False) -> torch.Tensor:
        """``words`` 32-bit integers of pinned memory to fill and hand to ``send``."""
        if not recorded:
            self.wait()
        if self._buffer is None or self._buffer.numel() < words:
            # (sizes differ from step to step: room for twice as many, so that they settle soon)
            self._buffer = torch.empty(max(2 * words, 64), dtype=torch.int32, pin_memory=True)
        return self._buffer[:words]

    def send(self, staged: torch.Tensor, dest: torch.Tensor, recorded: bool = False) -> None:
        """Queues the copy of what ``take`` gave to ``dest`` on the current stream."""
        dest.copy_(staged, non_blocking=True)
        if recorded:
            return
        if self._sent is None:
            self._sent = torch.cuda.Event()
        self._sent.record(torch.cuda.current_stream(dest.device))
