"""Shape-keyed pool of reusable output buffers.

Same contract as the reference's ``gpt_oss/triton/scratch_pool.py:17-22``: one
buffer per (shape, dtype, device); a later call with the same key returns the
same memory, so results are *borrowed* until the next such call. This is what
keeps a decode step free of allocations and therefore capturable in a HIP graph.
The pool of GPU buffers lives in ``csrc/host_ops.cpp``, where the ops take their outputs from it; buffers of other
devices, which need no library, are kept here.
"""
from __future__ import annotations

from operator import index
from typing import Any

import torch

from . import _lib

_pool: dict[tuple, torch.Tensor] = {}


def get(shape: tuple, dtype: torch.dtype, device: torch.device) -> torch.Tensor:
    shape, device = tuple(map(index, shape)), torch.device(device)
    if device.type == "cuda":
        buf = _lib.host().pool_get(shape, dtype, device)
        if buf is not None:                  # (None: a shape that only torch has an answer to)
            return buf
    key = (shape, dtype, device)
    buf = _pool.get(key)
    if buf is None:
        buf = _pool[key] = torch.empty(shape, dtype=dtype, device=device)
    return buf


def clear() -> None:
    _pool.clear()
    if _lib._host is not None:
        _lib._host.pool_clear()


def stats() -> dict[str, Any]:
    num_buffers, total_bytes = _lib._host.pool_stats() if _lib._host is not None else (0, 0)
    return {"num_buffers": num_buffers + len(_pool), "total_bytes": total_bytes + sum(t.numel() * t.element_size() for t in _pool.values())}
