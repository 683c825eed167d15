"""Small host arrays (key tables, descriptors) to the device in one copy."""
from __future__ import annotations

import numpy as np
import torch


class Staging:
    """One pinned buffer of an engine: ``open`` gives a new device buffer and
    the host bytes to fill, ``send`` copies them on the current stream without
    waiting.  A pageable copy waits for the device each time (14 us a copy, and
    the work queued before it); this takes 7.  The buffer is reused once its
    last copy is done; the device buffers are the caller's, and valid on the
    stream that was current."""

    def __init__(self, device: torch.device):
        self._device = device
        self._host: torch.Tensor | None = None
        self._bytes: np.ndarray | None = None
        self._sent: torch.cuda.Event | None = None
        self._dev: torch.Tensor | None = None

    def open(self, nbytes: int) -> tuple[torch.Tensor, np.ndarray]:
        if torch.cuda.is_current_stream_capturing():
            # a replay would copy what the buffer then holds
            raise RuntimeError("host values cannot be staged during stream capture")
        if self._sent is not None:
            self._sent.synchronize()
        if self._host is None or self._host.numel() < nbytes:
            self._host = torch.empty(max(4096, 2 * nbytes), dtype=torch.uint8, pin_memory=True)
            self._bytes = self._host.numpy()
        self._dev = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=self._device)
        return self._dev, self._bytes[:nbytes]

    def send(self) -> None:
        self._dev.copy_(self._host[: self._dev.numel()], non_blocking=True)
        if self._sent is None:
            self._sent = torch.cuda.Event()
        self._sent.record(torch.cuda.current_stream(self._device))
        self._dev = None

    def upload(self, array: np.ndarray) -> torch.Tensor:
        """The array's bytes as a device tensor (uint8)."""
        a = np.ascontiguousarray(array).reshape(-1).view(np.uint8)
        dev, host = self.open(a.size)
        host[:] = a
        self.send()
        return dev
