"""Host-side helpers shared by the two operators: length normalisation,
dtype codes, stream handles and the small int32 index arrays the C ABI takes."""
from __future__ import annotations

from array import array

import torch

from . import _lib

INT64_MAX = 9223372036854775807


def dtype_code(dt: torch.dtype, what: str, allow_f32: bool = False) -> int:
    if dt == torch.bfloat16:
        return _lib.DSA_DTYPE_BF16
    if dt == torch.float16:
        return _lib.DSA_DTYPE_F16
    if allow_f32 and dt == torch.float32:
        return _lib.DSA_DTYPE_F32
    raise ValueError(f"{what} dtype {dt} not supported (fp16/bf16{'/fp32' if allow_f32 else ''})")


def host_lengths(x, n: int | None = None, default: int | None = None) -> list[int]:
    """None -> [default]*n; list/tuple/ndarray/tensor -> list of ints (a device
    tensor is synchronised to the host, as the reference's .asnumpy() does)."""
    if x is None:
        return [int(default)] * int(n)
    if isinstance(x, torch.Tensor):
        return [int(v) for v in x.detach().to("cpu").reshape(-1).tolist()]
    return [int(v) for v in x]


def batch_lengths(x, n: int, default: int, name: str) -> list[int]:
    """host_lengths(x, n, default) as exactly n per-batch lengths: the kernels read one
    length per batch. A single value applies to every batch, as the reference's
    broadcast `zeros[B] + lengths` does (dense_loss_backward_triton.py:37-43,
    sparse_lightning_indexer_grad_kl_loss_triton.py:308-315); any other count raises."""
    v = host_lengths(x, n, default)
    if len(v) == 1 and n > 1:
        v = v * n
    if len(v) != n:
        raise ValueError(f"{name} must hold {n} per-batch lengths, got {len(v)}")
    return v


def per_batch_from_cumsum(cu: list[int]) -> list[int]:
    """TND cumulative actual_seq_lengths -> per-batch lengths
    (lightning_indexer_triton.py:294-296)."""
    out, prev = [], 0
    for c in cu:
        out.append(c - prev)
        prev = c
    return out


def prefix(lengths: list[int]) -> list[int]:
    out, acc = [0], 0
    for v in lengths:
        acc += v
        out.append(acc)
    return out


def require_device(*tensors: torch.Tensor) -> torch.device:
    dev = None
    for t in tensors:
        if t is None:
            continue
        if not isinstance(t, torch.Tensor) or t.device.type != "cuda":
            raise ValueError("inputs must be torch tensors on the GPU (HIP device)")
        if dev is None:
            dev = t.device
        elif t.device != dev:
            raise ValueError("all inputs must live on the same GPU")
    return dev


UPLOAD_MAX = 8192   # values a dsa_upload_i32 call takes


def upload(lib, device: torch.device, *arrays: list[int], zero: torch.Tensor | None = None, wait: bool = True):
    """The int32 length and offset arrays of a call on the device, views of one tensor (each padded
    to 16 bytes), written on the current stream by dsa_upload_i32 (one launch up to 56 values, then
    one per 960); `zero` (a byte tensor) is cleared by the first. For a device that is not the
    current one they go by a copy. With `wait` the host waits until the arrays and
    all that the caller put on this stream before are in place: a kept plan may run on any
    stream, and these arrays bound its addresses. A call that builds its plan and runs it at
    once, on one stream, needs no wait. Under stream capture there is none to wait for: the
    write is a node of the graph, and a plan built there runs in that graph."""
    flat, sizes = array("i"), []
    try:
        for a in arrays:
            flat.extend(a)
            pad = -len(flat) % 4
            if pad:
                flat.extend((0,) * pad)
            sizes.append(len(a) + pad)
    except OverflowError as e:   # torch's error for such a value
        raise RuntimeError("value cannot be converted to type int32 without overflow") from e
    n = len(flat)
    if device.index in (None, torch.cuda.current_device()):
        t = torch.empty(n, dtype=torch.int32, device=device)
        src, dst, stream = flat.buffer_info()[0], t.data_ptr(), stream_ptr(device)
        zero_ptr, zero_bytes = ptr(zero), 0 if zero is None else zero.numel()
        for i in range(0, max(n, 1), UPLOAD_MAX):
            _lib.check(lib.dsa_upload_i32(src + 4 * i, min(n - i, UPLOAD_MAX), dst + 4 * i, zero_ptr, zero_bytes,
                                          stream), "dsa_upload_i32")
            zero_ptr, zero_bytes = None, 0
    else:
        if zero is not None:
            zero.zero_()
        t = torch.frombuffer(flat, dtype=torch.int32).to(device) if n else torch.empty(0, dtype=torch.int32, device=device)
    if wait and not torch.cuda.is_current_stream_capturing():
        torch.cuda.current_stream(device).synchronize()
    return t.split(sizes)


def stream_ptr(device: torch.device) -> int:
    # the raw handle, without the Stream object that torch.cuda.current_stream builds (2.5 us a call)
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if device.index is None else device.index)


def ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()
