"""Calls into libq6moe.so on a device's current stream.

Small operators are bound by this host path (a 4-token projection's kernel
takes 5 us), so it stays short: the device guard only where another device is
current, the raw stream handle without a Stream object, pointers as plain
integers (ctypes converts them by the declared argument types).
"""

import torch

from . import _lib

def run(what, fn, device, *args):
    """``fn(*args, stream)`` with ``device`` (a GPU tensor's, so with an index) current; raises on an error code."""
    if device.type != "cuda":
        raise ValueError(f"Expected a cuda device, but got: {device}")
    index = device.index
    # looked up per call: a torch built without a GPU backend lacks both names, and
    # still imports the package
    raw_stream = torch._C._cuda_getCurrentRawStream
    if index == torch._C._cuda_getDevice():
        rc = fn(*args, raw_stream(index))
    else:
        with torch.cuda.device(index):
            rc = fn(*args, raw_stream(index))
    if rc:
        _lib.check(rc, what)
