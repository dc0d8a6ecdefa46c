"""Shape-keyed pool of reusable output buffers.

Same contract as the reference's ``gpt_oss/triton/scratch_pool.py:17-22``: one
buffer per (shape, dtype, device); a later call with the same key returns the
same memory, so results are *borrowed* until the next such call. This is what
keeps a decode step free of allocations and therefore capturable in a HIP graph.
The pool itself lives in ``csrc/host_ops.cpp``, where the ops take their outputs from it.
"""
from __future__ import annotations

from operator import index
from typing import Any

import torch

from ._lib import host


def get(shape: tuple, dtype: torch.dtype, device: torch.device) -> torch.Tensor:
    return host().pool_get(tuple(map(index, shape)), dtype, torch.device(device))


def clear() -> None:
    host().pool_clear()


def stats() -> dict[str, Any]:
    num_buffers, total_bytes = host().pool_stats()
    return {"num_buffers": num_buffers, "total_bytes": total_bytes}
