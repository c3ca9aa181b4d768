"""Device plumbing: torch tensors as device buffers and the current HIP stream."""
import torch

from . import _lib

DTYPES = {torch.float32: _lib.DT_F32, torch.float16: _lib.DT_F16, torch.bfloat16: _lib.DT_BF16}
TORCH = {v: k for k, v in DTYPES.items()}


def ptr(t):
    return None if t is None else t.data_ptr()


def stream():
    """The current HIP stream's handle (as torch.cuda.current_stream().cuda_stream, whose Stream object
    alone costs 2.6 us a call)."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def device_f32(t, like):
    """t as contiguous fp32 on like's device (None: None)."""
    if t is None or (t.dtype is torch.float32 and t.device == like.device and t.is_contiguous()):
        return t
    return t.to(device=like.device, dtype=torch.float32).contiguous()


def require_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise ValueError("tensors must be on the GPU")
