"""What every kernel wrapper does around its C call, kept short: a small launch
is bound by the host, where a device guard, a stream object and ctypes arrays
built per call cost more than the kernel runs.
"""

from __future__ import annotations

import torch

_current_device = torch.cuda.current_device


def _stream_handle(index: int) -> int:
    return torch.cuda.current_stream(index).cuda_stream


# The current stream's handle without building a Stream object.
raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", _stream_handle)


def launch(index: int, entry, *args) -> int:
    """``entry(*args, stream)`` with device ``index`` current and its current
    stream; returns the status."""
    if _current_device() == index:
        return entry(*args, raw_stream(index))
    with torch.cuda.device(index):
        return entry(*args, raw_stream(index))


def query(index: int, entry, *args):
    """``entry(*args)`` with device ``index`` current."""
    if _current_device() == index:
        return entry(*args)
    with torch.cuda.device(index):
        return entry(*args)


def vector_ready(t: torch.Tensor) -> bool:
    """Rows of a 4-D tensor start on 16-byte boundaries (128-bit accesses)."""
    s = t.stride()
    return not (t.data_ptr() | (s[0] | s[1] | s[2]) * t.element_size()) & 15
