"""The looped column's copy-forward bookkeeping on MI355X.

``end_pass`` is what the column's pass loop runs (``vsp_pass_end``): the halting bookkeeping, the
tokens halting now freezing their projections into the carried ones (``vesper/loop.py:523-537``,
``_merge``), the hidden state of the tokens still in the loop (``vesper/loop.py:441-452``) and the next
pass's norm, in one launch. ``halt_step`` and ``residual_rows_where`` are two of its parts as launches of
their own, for the loop with ``where`` merges and the decoder's last add.

``copy_rows_where(items)`` performs, for each ``(src, dst, flags)``, ``dst[flags] = src[flags]``
over the leading ``[b, n]`` token dimensions, every item in one kernel launch
(``vsp_copy_rows_where``): the freezing alone, for a caller with a pass loop of its own (the package's
loop does not call it). Only flagged rows are read and written.
"""

from __future__ import annotations

import ctypes
from collections.abc import Sequence

import torch
from torch import Tensor

from vesper.contracts import ContractError
from vesper.kernels import _lib

MAX_ITEMS = 8  # tensors per launch


def copy_rows_where(items: Sequence[tuple[Tensor, Tensor, Tensor]]) -> None:
    """``dst[flags] = src[flags]`` in place for each ``(src, dst, flags)``, one launch for all.

    Args:
        items: up to eight triples on one GPU: ``src`` and ``dst`` of one shape and dtype with
            leading dimensions ``[b, n]`` (``dst`` contiguous: it is written in place), ``flags``
            bool ``[b, n]``; every item has the same ``b * n``.

    Raises:
        ContractError: on more than eight items, shapes, dtypes or devices that disagree, or a
            ``dst`` that is not contiguous.
    """
    if len(items) > MAX_ITEMS:
        raise ContractError(f"{len(items)} tensors: at most {MAX_ITEMS} per launch")
    if not items:
        return
    device = items[0][1].device
    rows = None
    srcs, dsts, flags, sizes = [], [], [], []
    for i, (src, dst, flag) in enumerate(items):
        if src.shape != dst.shape or src.dtype != dst.dtype:
            raise ContractError(f"item {i}: src {tuple(src.shape)} {src.dtype}, dst {tuple(dst.shape)} {dst.dtype}")
        if flag.dtype != torch.bool or flag.dim() != 2 or tuple(dst.shape[:2]) != tuple(flag.shape):
            raise ContractError(f"item {i}: flags must be bool {tuple(dst.shape[:2])}, got {tuple(flag.shape)} {flag.dtype}")
        if any(t.device != device for t in (src, dst, flag)) or device.type != "cuda":
            raise ContractError(f"item {i}: every tensor must be on one GPU ({device})")
        if not dst.is_contiguous():
            raise ContractError(f"item {i}: dst must be contiguous (it is written in place)")
        n_rows = flag.numel()
        if rows is None:
            rows = n_rows
        elif rows != n_rows:
            raise ContractError(f"item {i}: {n_rows} token rows, the first item has {rows}")
        src_c, flag_c = src.contiguous(), flag.contiguous()
        srcs.append(src_c)
        dsts.append(dst)
        flags.append(flag_c)
        sizes.append(dst.numel() * dst.element_size() // max(n_rows, 1))
    count = len(items)
    src_arr = (ctypes.c_void_p * count)(*[t.data_ptr() for t in srcs])
    dst_arr = (ctypes.c_void_p * count)(*[t.data_ptr() for t in dsts])
    flag_arr = (ctypes.c_void_p * count)(*[t.data_ptr() for t in flags])
    size_arr = (ctypes.c_size_t * count)(*sizes)
    with _lib.on_device(device):
        _lib.call("vsp_copy_rows_where", count, ctypes.cast(src_arr, ctypes.c_void_p),
                  ctypes.cast(dst_arr, ctypes.c_void_p), ctypes.cast(size_arr, ctypes.c_void_p),
                  ctypes.cast(flag_arr, ctypes.c_void_p), int(rows or 0), _lib.stream_of(device))


def halt_step(active: Tensor, exits: Tensor | None, n_iters: Tensor) -> tuple[Tensor, Tensor]:
    """One pass's halting bookkeeping in one launch (``vsp_halt_step``): ``halts = active & exits``
    (every active token when ``exits`` is None, the last pass), ``n_iters += active`` in place, and
    the next pass's ``active & ~halts``; returns ``(halts, next_active)``.

    Args:
        active: bool ``[b, n]``; exits: bool ``[b, n]`` or None; n_iters: contiguous int32 ``[b, n]``.

    Raises:
        ContractError: on shapes, dtypes or devices that disagree.
    """
    shape = tuple(active.shape)
    if active.dtype != torch.bool or active.device.type != "cuda":
        raise ContractError(f"active: bool on CUDA, got {active.dtype} on {active.device}")
    if exits is not None and (tuple(exits.shape) != shape or exits.dtype != torch.bool or exits.device != active.device):
        raise ContractError(f"exits: bool {shape} on {active.device}")
    if (tuple(n_iters.shape) != shape or n_iters.dtype != torch.int32 or n_iters.device != active.device
            or not n_iters.is_contiguous()):
        raise ContractError(f"n_iters: contiguous int32 {shape} on {active.device}")
    a = active.contiguous()
    e = None if exits is None else exits.contiguous()
    halts = torch.empty_like(a)
    nxt = torch.empty_like(a)
    with _lib.on_device(active.device):
        _lib.call("vsp_halt_step", a.data_ptr(), _lib.ptr(e), n_iters.data_ptr(), halts.data_ptr(), nxt.data_ptr(),
                  a.numel(), _lib.stream_of(active.device))
    return halts, nxt


def residual_rows_where(x1: Tensor, a: Tensor, x: Tensor, flags: Tensor | None) -> None:
    """``x[r] = x1[r] + a[r]`` in place for the token rows with ``flags[r]`` set (every row when
    ``flags`` is None), one launch (``vsp_residual_rows_where``): the residual add after a pass's
    attention written straight into the loop's hidden state, only for the tokens still in the
    loop (``vesper/loop.py:452``).

    Args:
        x1: float32 ``[b, n, d]``; a: bfloat16 ``[b, n, d]`` (added in float32); x: contiguous
            float32 ``[b, n, d]``, written in place (not ``x1``); flags: bool ``[b, n]`` or None.

    Raises:
        ContractError: on shapes, dtypes or devices that disagree.
    """
    if x1.dim() != 3 or x1.dtype != torch.float32 or x1.device.type != "cuda":
        raise ContractError(f"x1: float32 [b, n, d] on CUDA, got {tuple(x1.shape)} {x1.dtype} on {x1.device}")
    if a.shape != x1.shape or a.dtype != torch.bfloat16 or a.device != x1.device:
        raise ContractError(f"a: bf16 {tuple(x1.shape)}, got {tuple(a.shape)} {a.dtype}")
    if x.shape != x1.shape or x.dtype != torch.float32 or x.device != x1.device or not x.is_contiguous():
        raise ContractError(f"x: contiguous float32 {tuple(x1.shape)} on {x1.device}")
    if x.data_ptr() == x1.data_ptr():
        raise ContractError("x must not be x1")
    if flags is not None and (tuple(flags.shape) != tuple(x1.shape[:2]) or flags.dtype != torch.bool
                              or flags.device != x1.device):
        raise ContractError(f"flags: bool {tuple(x1.shape[:2])} on {x1.device}")
    x1c, ac = x1.contiguous(), a.contiguous()
    for name, t in (("x1", x1c), ("a", ac), ("x", x)):
        if t.data_ptr() % 16:
            raise ContractError(f"{name} must be 16-byte aligned")
    fl = None if flags is None else flags.contiguous().view(torch.uint8)
    b, n, d = x1.shape
    with _lib.on_device(x1.device):
        _lib.call("vsp_residual_rows_where", x1c.data_ptr(), ac.data_ptr(), x.data_ptr(), _lib.ptr(fl), b * n, d,
                  _lib.stream_of(x1.device))


def end_pass(x1: Tensor, a: Tensor, x: Tensor, active: Tensor, exits: Tensor | None, n_iters: Tensor,
             freeze: Sequence[tuple[Tensor, Tensor]], *, norm: bool) -> tuple[Tensor, Tensor | None]:
    """The end of a looped column's pass in one launch (``vsp_pass_end``): ``halt_step``, then
    ``copy_rows_where`` of each ``(src, dst)`` of ``freeze`` where a token halts, then
    ``residual_rows_where(x1, a, x, active)``, then, with ``norm``, ``rms_norm_bf16(x)``; bitwise those
    launches' results.

    Args:
        x1: float32 ``[b, n, d]``; a: bfloat16 ``[b, n, d]``; x: contiguous float32 ``[b, n, d]``,
            written in place (not ``x1``); ``d`` a multiple of 8 in 8..2048.
        active, exits: bool ``[b, n]`` (``exits`` None: the last pass); n_iters: contiguous int32
            ``[b, n]``, counted up in place.
        freeze: up to eight pairs of one shape and dtype, leading ``[b, n]``, the second contiguous
            (written in place).

    Returns:
        the next pass's active flags and its normalized input (None without ``norm``).

    Raises:
        ContractError: on shapes, dtypes, devices or layouts outside that contract.
    """
    lead, device = x1.shape[:2], x1.device
    if x1.dim() != 3 or x1.dtype != torch.float32 or device.type != "cuda":
        raise ContractError(f"x1: float32 [b, n, d] on CUDA, got {tuple(x1.shape)} {x1.dtype} on {device}")
    for name, t, dtype, shape in (("a", a, torch.bfloat16, x1.shape), ("x", x, torch.float32, x1.shape),
                                  ("active", active, torch.bool, lead), ("n_iters", n_iters, torch.int32, lead),
                                  ("exits", exits, torch.bool, lead)):
        if t is not None and (t.dtype != dtype or t.shape != shape or t.device != device):
            raise ContractError(f"{name}: {dtype} {tuple(shape)} on {device}, got {tuple(t.shape)} {t.dtype} on {t.device}")
    if len(freeze) > MAX_ITEMS:
        raise ContractError(f"{len(freeze)} tensors: at most {MAX_ITEMS} per launch")
    for i, (src, dst) in enumerate(freeze):
        if src.shape != dst.shape or src.dtype != dst.dtype or src.shape[:2] != lead or src.device != device or dst.device != device:
            raise ContractError(f"item {i}: src {tuple(src.shape)} {src.dtype}, dst {tuple(dst.shape)} {dst.dtype}")
    if not all(t.is_contiguous() for t in (x, n_iters, *(dst for _, dst in freeze))):
        raise ContractError("x, n_iters and every freeze target must be contiguous (they are written in place)")
    b, n, d = x1.shape
    if d % 8 or not 8 <= d <= 2048:
        raise ContractError(f"x1: width {d} is not a multiple of 8 in 8..2048")
    x1, a, active = x1.contiguous(), a.contiguous(), active.contiguous()
    exits_c = None if exits is None else exits.contiguous()
    sources = [src.contiguous() for src, _ in freeze]
    for name, t in (("x1", x1), ("a", a), ("x", x)):
        if t.data_ptr() % 16:
            raise ContractError(f"{name} must be 16-byte aligned")
    rows, count = b * n, len(freeze)
    if rows and x.data_ptr() == x1.data_ptr():
        raise ContractError("x must not be x1")
    nxt = torch.empty_like(active)
    out = torch.empty(b, n, d, dtype=torch.bfloat16, device=device) if norm else None
    if rows == 0:
        return nxt, out
    pointers = ctypes.c_void_p * count
    srcs, dsts = pointers(*[s.data_ptr() for s in sources]), pointers(*[t.data_ptr() for _, t in freeze])
    sizes = (ctypes.c_size_t * count)(*[t.numel() * t.element_size() // rows for _, t in freeze])
    with _lib.on_device(device):
        _lib.call("vsp_pass_end", count, ctypes.cast(srcs, ctypes.c_void_p), ctypes.cast(dsts, ctypes.c_void_p),
                  ctypes.cast(sizes, ctypes.c_void_p), x1.data_ptr(), a.data_ptr(), x.data_ptr(), active.data_ptr(),
                  _lib.ptr(exits_c), n_iters.data_ptr(), nxt.data_ptr(), _lib.ptr(out), rows, d, _lib.stream_of(device))
    return nxt, out
