"""Affine (MLX) quantized projections and the Hadamard rotation on MI355X.

Mirrors hadamardRotate and the rotated PackedLinear forward (Sources/IshizukiKit/Core/
Hadamard.swift:8-23,180-231) and VerifyMatmul.apply/applyAny (Core/VerifyMatmul.swift:63-120)
over libishizuki_hip. Kernel calls return None when declined, like the reference's nil.
"""
import torch

from . import _lib
from ._torch import DTYPES, device_f32, ptr, require_cuda, stream

supported_rows = range(2, 9)   # VerifyMatmul.supportedRows (:12)


def minimum_rows(nbytes):
    """VerifyMatmul.minimumRows (Core/VerifyMatmul.swift:19-26), re-measured on MI355X.

    The reference's thresholds (2 rows from 100 MB, 3 from 10 MB, 4 from 5 MB, else 6) are where
    its verify kernel beats MLX's per-row path on an M1 Max. Here the alternative is M one-row
    GEMV calls, and one M-row verify call is faster from M = 2 at every size measured (1.6 MB
    attention k/v to the 397 MB vocabulary head, `python bench.py --policy`), so the minimum is 2.
    """
    return 2


def hadamard_rotate(x, block, signs=None, inverse=False):
    """hadamardRotate: y = WHT_block(x * signs)/sqrt(block) in fp32, cast back to x.dtype."""
    require_cuda(x)
    shape = x.shape
    x2 = x.reshape(-1, shape[-1]).contiguous()
    y = torch.empty_like(x2)
    s = device_f32(signs, x)
    rc = _lib.lib().ishz_hadamard(ptr(x2), DTYPES.get(x.dtype, -1), x2.shape[0], x2.shape[1], block,
                                  ptr(s), int(inverse), ptr(y), stream())
    if not _lib.check(rc, "hadamard"):
        raise ValueError(_lib.last_error())
    return y.reshape(shape)


def _check_width(N, K, x, weight, scales, biases, group_size, bits):
    """The C calls take K from x and step through the pack by it, so a pack of another width would be read
    past its end, or in the wrong rows. What they decline is left to them. (A pack that fits is told first: 0.6 us.)"""
    n = N * K
    if (scales.numel() * group_size == n and biases.numel() * group_size == n
            and weight.numel() * weight.element_size() * 8 == n * bits):
        return
    if (x.dtype not in DTYPES or scales.dtype not in (torch.float16, torch.bfloat16) or not 2 <= bits <= 8
            or group_size < 32 or group_size % 32 or K % group_size or K % 128):
        return
    raise _lib.IshzError(f"x of width {K} through a {bits}-bit pack of {N} rows of width "
                         f"{scales.numel() // max(N, 1) * group_size}")


def quantized_matmul(x, weight, scales, biases, group_size=64, bits=2):
    """y = x . dequant(weight)^T for x [M, K], M in 1..16; None if declined."""
    require_cuda(x, weight, scales, biases)
    x = x.contiguous()
    M, K = x.shape
    N = weight.shape[0]
    _check_width(N, K, x, weight, scales, biases, group_size, bits)
    y = torch.empty((M, N), dtype=x.dtype, device=x.device)
    rc = _lib.lib().ishz_affine_matmul(x.data_ptr(), DTYPES.get(x.dtype, -1), M, K, weight.data_ptr(), scales.data_ptr(),
                                       biases.data_ptr(), DTYPES.get(scales.dtype, -1), N, bits, group_size, y.data_ptr(),
                                       stream())
    return y if _lib.check(rc, "affine_matmul") else None


def verify_apply(x, weight, scales, biases, group_size=64, bits=2):
    """VerifyMatmul.apply: declines below the weight's minimum row count (and above 8)."""
    if x.dim() != 2 or x.shape[0] not in supported_rows:
        return None
    if x.shape[0] < minimum_rows(weight.numel() * weight.element_size()):
        return None
    return quantized_matmul(x, weight, scales, biases, group_size, bits)


def linear(x, weight, scales, biases, signs=None, block=0, group_size=64, bits=2, _prestage=True):
    """Rotated PackedLinear forward: rotate (fused for one row) then the quantized matmul.

    With block <= 128 and more than two rows the workspace holds every row's x rotated and staged
    once for all workgroups (with one or two rows each workgroup rotates x itself, which measured
    faster); `_prestage=False` passes none, so each workgroup rotates x itself at any row count
    (test hook; the general path for other blocks needs the workspace)."""
    require_cuda(x, weight, scales, biases)
    x = x.contiguous()
    M, K = x.shape
    N = weight.shape[0]
    _check_width(N, K, x, weight, scales, biases, group_size, bits)
    y = torch.empty((M, N), dtype=x.dtype, device=x.device)
    L = _lib.lib()
    if M > 1 and x.dtype is torch.bfloat16:  # their fp16 image
        needs = True
    elif block:  # (one fp16 row of a 2-bit pack is rotated and staged in the GEMV)
        needs = _prestage and not (M == 1 and bits == 2 and group_size in (64, 128) and x.dtype is torch.float16)
    else:
        needs = False
    ws_bytes = L.ishz_affine_workspace_size(M, K) if needs else 0
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device) if ws_bytes else None
    s = device_f32(signs, x) if block else None
    rc = L.ishz_affine_linear(x.data_ptr(), DTYPES.get(x.dtype, -1), M, K, ptr(s), block, weight.data_ptr(),
                              scales.data_ptr(), biases.data_ptr(), DTYPES.get(scales.dtype, -1), N, bits, group_size,
                              y.data_ptr(), ptr(ws), ws_bytes, stream())
    return y if _lib.check(rc, "affine_linear") else None


def linear_rows(x, weight, scales, biases, signs=None, block=0, group_size=64, bits=2):
    """The rotated PackedLinear forward for a prompt: any number of rows in one call; None if
    declined (fp32 x, odd widths, other groups), where `linear` takes 16 rows at a time."""
    require_cuda(x, weight, scales, biases)
    x = x.contiguous()
    M, K = x.shape
    N = weight.shape[0]
    _check_width(N, K, x, weight, scales, biases, group_size, bits)
    L = _lib.lib()
    # what the library declines by these is declined before anything is allocated
    takes = (K % 256 == 0 and (x.dtype is torch.float16 or x.dtype is torch.bfloat16) and bits in (2, 4, 6, 8)
             and (group_size == 64 or group_size == 128))
    ws_bytes = L.ishz_affine_rows_workspace_size(M, K, N) if takes else 0
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device) if takes else None
    y = torch.empty((M, N), dtype=x.dtype, device=x.device) if takes else None
    s = device_f32(signs, x) if block else None
    rc = L.ishz_affine_linear_rows(x.data_ptr(), DTYPES.get(x.dtype, -1), M, K, ptr(s), block, weight.data_ptr(),
                                   scales.data_ptr(), biases.data_ptr(), DTYPES.get(scales.dtype, -1), N, bits, group_size,
                                   ptr(y), ptr(ws), ws_bytes, stream())
    return y if _lib.check(rc, "affine_linear_rows") else None
