"""ctypes plumbing shared by the case ``op`` modules.

Each case library exports plain C functions (see the headers in include/):
device pointers as ``void*``, sizes as ``int64_t``, the HIP stream as a
pointer, and an ``int`` status (0 = success).  ``bind`` attaches argument
and result types; ``check`` turns a non-zero status into the RuntimeError
the reference's TORCH_CHECK failures would have raised.
"""

import ctypes
import os

import torch

c_void_p = ctypes.c_void_p
c_int64 = ctypes.c_int64
c_int = ctypes.c_int
c_float = ctypes.c_float
c_size_t = ctypes.c_size_t
c_double = ctypes.c_double


def bind(lib, name, argtypes, restype=ctypes.c_int):
    fn = getattr(lib, name)
    fn.argtypes = argtypes
    fn.restype = restype
    return fn


def bind_last_error(lib, name):
    fn = getattr(lib, name)
    fn.argtypes = []
    fn.restype = ctypes.c_char_p
    return fn


def check(status, last_error, what):
    if status != 0:
        msg = last_error().decode(errors="replace")
        raise RuntimeError(f"{what}: {msg} (status {status})")


def ptr(t):
    """Device address of a tensor (0 for an empty tensor)."""
    return ctypes.c_void_p(t.data_ptr() if t.numel() else 0)


def stream_of(t):
    """The current torch stream of the tensor's device, as a HIP stream handle."""
    return ctypes.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


_current_device = getattr(torch._C, "_cuda_getDevice", None)
_current_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def launch(fn, device, *args):
    """``fn(*args, stream)``: a C entry on GPU ``device`` (an index), enqueued on
    torch's current stream of that device, which is made the current device
    for the call.

    An op's body is a few microseconds of Python around one call, and a
    training step runs two of them, one in autograd's worker thread: the
    device guard, the Stream object and a ctypes object per pointer were most
    of it (RBF training step at 256 x 256: 117 -> 84 us with the checks and
    allocations written for their common case).  Pointers are passed as the
    integers ``data_ptr()`` returns.
    """
    if _current_device() == device:
        return fn(*args, _current_raw_stream(device))
    with torch.cuda.device(device):
        return fn(*args, _current_raw_stream(device))


def scratch(like, best, least):
    """A workspace of ``best`` bytes beside the float32 tensor ``like``, or of
    ``least`` where that does not fit: (tensor, bytes).  For calls that run with
    less, if slower."""
    try:
        return like.new_empty((max(best, 8) + 3) // 4), best
    except torch.OutOfMemoryError:
        if least >= best:
            raise
    return like.new_empty((max(least, 8) + 3) // 4), least


def require(cond, msg):
    """TORCH_CHECK equivalent for the Python boundary."""
    if not cond:
        raise RuntimeError(msg)


def checking():
    """True when NL2K_CHECK=1: ops then also read the status words their
    kernels leave in the workspace (a synchronisation per call)."""
    return os.environ.get("NL2K_CHECK", "") == "1"
