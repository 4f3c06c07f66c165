"""Copy one request's prefix across every plane of a packed KV arena on the GPU.

Drop-in for ``copy_packed_prefix`` (qwen3_tts_engine/packed_kv.py:6-31): the same
arguments, the same validation and ``ValueError`` raised before any device write; the copy
itself is the ``q3t_copy_strided`` HIP kernel (bit-exact element copy, any strides).
"""
import math

import torch

from . import _lib


def _is_index(value) -> bool:
    return type(value) is int


def copy_packed_prefix(target, source, slot, row=0, length=None):
    """target[:, slot, :, :length] = source[:, row, :, :length]; other slots and the tail
    of the selected slot are preserved."""
    if (
        not isinstance(target, torch.Tensor)
        or not isinstance(source, torch.Tensor)
        or target.ndim != 5
        or source.ndim != 5
        or any(size <= 0 for size in (*target.shape, *source.shape))
        or (target.shape[0], target.shape[2], target.shape[4])
        != (source.shape[0], source.shape[2], source.shape[4])
        or target.device != source.device
        or target.dtype != source.dtype
        or target.untyped_storage().data_ptr() == source.untyped_storage().data_ptr()
    ):
        raise ValueError("Expected independent compatible packed KV tensors")
    length = source.shape[3] if length is None else length
    if (
        not _is_index(slot) or not 0 <= slot < target.shape[1]
        or not _is_index(row) or not 0 <= row < source.shape[1]
        or not _is_index(length) or not 0 < length <= min(target.shape[3], source.shape[3])
    ):
        raise ValueError("Expected a valid packed KV row and prefix length")
    copy_rows(target[:, slot, :, :length], source[:, row, :, :length])


def copy_rows(dst: torch.Tensor, src: torch.Tensor) -> None:
    """Element copy dst <- src of equal shape (<= 5 dims, any strides) by the HIP kernel."""
    if dst.shape != src.shape or dst.dtype != src.dtype:
        raise ValueError("copy requires equal shapes and dtypes")
    if dst.ndim > 5 or dst.ndim == 0:
        raise ValueError("copy supports 1 to 5 dimensions")
    device = _lib.require_gpu(dst, src)
    if dst.numel() == 0:
        return
    n = dst.ndim
    sizes = (_lib.c_i64 * n)(*dst.shape)
    ds = (_lib.c_i64 * n)(*dst.stride())
    ss = (_lib.c_i64 * n)(*src.stride())
    status = _lib.library().q3t_copy_strided(dst.data_ptr(), src.data_ptr(), dst.element_size(),
                                             n, sizes, ds, ss, _lib.stream_handle(device))
    _lib.check(status, "copy_rows")


def grow_blocks(dst: torch.Tensor, src: torch.Tensor, used: int) -> None:
    """dst (planes, slots, heads, new, width) <- src (planes, slots, heads, old, width), old <= new:
    the rows of slots below ``used``, then zeros; every element of dst is written.  Both
    contiguous, and rows as the kernel takes them (``can_grow_blocks``)."""
    device = _lib.require_gpu(dst, src)
    planes, slots, heads, rows, width = dst.shape
    size = dst.element_size() * width
    status = _lib.library().q3t_grow_arena(dst.data_ptr(), src.data_ptr(), planes, slots, used, heads,
                                           src.shape[3] * size, rows * size, _lib.stream_handle(device))
    _lib.check(status, "grow_blocks")


def can_grow_blocks(dst: torch.Tensor, src: torch.Tensor) -> bool:
    size = dst.element_size() * dst.shape[-1]
    return (dst.is_cuda and dst.numel() > 0 and src.numel() > 0 and dst.dtype == src.dtype and dst.is_contiguous()
            and src.is_contiguous() and dst.data_ptr() % 16 == 0 and src.data_ptr() % 16 == 0
            and (src.shape[-2] * size) % 16 == 0 and (dst.shape[-2] * size) % 16 == 0
            and grow_launch_fits(math.prod(dst.shape[:-2]), dst.shape[-2] * size))


def grow_launch_fits(blocks: int, block_bytes: int) -> bool:
    """Whether one launch covers the blocks: 1024 16-byte vectors a workgroup of 256 threads, fewer
    than 2^32 threads, 32-bit vector numbers within a block."""
    vectors = block_bytes // 16
    return vectors < 1 << 31 and blocks * -(-vectors // 1024) < 1 << 24
