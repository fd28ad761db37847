"""``fps``: drop-in for ``torch_cluster.fps`` (reference:
``torch_cluster/fps.py:35-108``), on GPU tensors and on CPU tensors.

Same signature, defaults and argument handling; stays ``torch.jit.script``-
able.  The sampling itself is ``torch.ops.torch_cluster.fps``, registered by
this package's native library.
"""
from typing import List, Optional, Union

import torch
from torch import Tensor

from ._segments import batch_pointers, examples_or_unknown


@torch.jit._overload  # noqa
def fps(src, batch, ratio, random_start, batch_size, ptr):  # noqa
    # type: (Tensor, Optional[Tensor], Optional[float], bool, Optional[int], Optional[Tensor]) -> Tensor  # noqa
    pass  # pragma: no cover


@torch.jit._overload  # noqa
def fps(src, batch, ratio, random_start, batch_size, ptr):  # noqa
    # type: (Tensor, Optional[Tensor], Optional[Tensor], bool, Optional[int], Optional[Tensor]) -> Tensor  # noqa
    pass  # pragma: no cover


@torch.jit._overload  # noqa
def fps(src, batch, ratio, random_start, batch_size, ptr):  # noqa
    # type: (Tensor, Optional[Tensor], Optional[float], bool, Optional[int], Optional[List[int]]) -> Tensor  # noqa
    pass  # pragma: no cover


@torch.jit._overload  # noqa
def fps(src, batch, ratio, random_start, batch_size, ptr):  # noqa
    # type: (Tensor, Optional[Tensor], Optional[Tensor], bool, Optional[int], Optional[List[int]]) -> Tensor  # noqa
    pass  # pragma: no cover


def fps(  # noqa
    src: torch.Tensor,
    batch: Optional[Tensor] = None,
    ratio: Optional[Union[Tensor, float]] = None,
    random_start: bool = True,
    batch_size: Optional[int] = None,
    ptr: Optional[Union[Tensor, List[int]]] = None,
):
    r"""Farthest point sampling: per example, starting from one row, the row
    farthest from the rows sampled so far is added until ``ceil(ratio * N)``
    rows are chosen.

    Args:
        src: points, ``[N, F]``.
        batch: ``[N]`` example vector.
        ratio: sampling ratio, a float, a scalar tensor or one value per
            example (default 0.5).
        random_start: start from a random row of every example instead of its
            first.
        batch_size: number of examples (saves a device-to-host read).
        ptr: example boundaries in CSR form (tensor or list) instead of
            ``batch``.

    Returns the int64 row numbers of the samples, example after example, in
    sampling order.
    """
    # fp32 rows with a plain ratio: pointers and numbers of samples on the
    # device, without torch calls
    if (ptr is None and src.is_cuda and src.dtype == torch.float32
            and src.numel() > 0
            and (batch_size is None or batch_size > 0)):
        share_of: float = -1.0
        if ratio is None:
            share_of = 0.5
        elif isinstance(ratio, float):
            share_of = ratio
        if share_of > 0.0 and share_of <= 1.0:
            if batch is not None:
                assert src.size(0) == batch.numel()
            return torch.ops.pytorch_cluster_amd.fps_batched(
                src, batch, examples_or_unknown(batch_size), share_of,
                random_start)

    # the share of every example that is sampled, as the operator takes it: a
    # tensor (TorchScript resolves the three cases per overload, in this
    # order)
    if ratio is None:
        share = torch.full((), 0.5, dtype=src.dtype, device=src.device)
    elif isinstance(ratio, float):
        share = torch.full((), ratio, dtype=src.dtype, device=src.device)
    else:
        share = ratio

    # example boundaries, whichever way the caller states them
    if ptr is not None:
        if isinstance(ptr, list):
            bounds = torch.tensor(ptr, dtype=torch.long, device=src.device)
        else:
            bounds = ptr
    elif batch is not None:
        bounds = batch_pointers(src, batch, batch_size)
    else:
        bounds = torch.tensor([0, src.size(0)], dtype=torch.long,
                              device=src.device)
    return torch.ops.torch_cluster.fps(src, bounds, share, random_start)
