"""Whole numbers of a step on their way to the device, in stream order and without waiting for it."""
from __future__ import annotations

import torch


def upload(values, device) -> torch.Tensor:
    """`values` as an int32 tensor on the device.  They travel through pinned memory: a copy from ordinary memory returns
    when the stream has run up to it, so that every step waited for the one before and the device for its host (steps of
    2,048 tokens through four layers with experts, one behind the other, 2,592 -> 2,412 us each).  torch's allocator of pinned
    memory gives the memory out again when the copy has run; so it cannot be captured: a replay would copy whatever is there by then."""
    host = torch.as_tensor(values, dtype=torch.int32)
    if torch.device(device).type != "cuda":
        return host.to(device)
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("upload: numbers from the host cannot be captured into a graph")
    return host.pin_memory().to(device, non_blocking=True)
