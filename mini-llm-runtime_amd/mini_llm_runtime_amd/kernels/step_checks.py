"""The device-side checks of a step's metadata as one launch and one transfer
(``mlr_check_step``), where torch operations take a launch per comparison.

``step_flags`` returns the flags of everything it was given; the callers raise
the reference's errors from them, in the reference's order. It takes int64
tensors on one HIP device and returns None for what the kernel does not take
(other devices, many tokens): the caller then evaluates its torch operations.
"""

from __future__ import annotations

import torch

from .. import _lib

# enum mlr_check_flags in include/mlr_attn.h
CONTEXT, WIDTH, BLOCK = 1, 2, 4
QSL_START, QSL_ORDER, QSL_END, QUERY_LEN, COVER = 8, 16, 32, 64, 128
SLOT_RANGE, POSITION, SLOT, REPEAT = 256, 512, 1024, 2048
DECODE_SHIFT = 3


def step_flags(block_size: int, num_blocks: int, *, tables: torch.Tensor | None = None,
               ctx: torch.Tensor | None = None, qsl: torch.Tensor | None = None,
               positions: torch.Tensor | None = None, slots: torch.Tensor | None = None,
               decoding: torch.Tensor | None = None, max_query_len: int = 0,
               detail: bool = False):
    """The flags (and, with ``detail``, the host copies of query_start_loc,
    context_lens and the per-request invalid-block words) or None."""
    given = [t for t in (tables, ctx, qsl, positions, slots) if t is not None]
    device = given[0].device
    if device.type != "cuda" or block_size <= 0 or num_blocks <= 0:
        return None
    for t in given:
        if t.dtype is not torch.long or t.device != device:
            return None
    reqs = 0 if ctx is None else ctx.shape[0]
    tokens = 0 if slots is None else slots.shape[0]
    if ((ctx is not None and (ctx.ndim != 1 or tables is None or tables.ndim != 2
                              or tables.shape[0] != reqs))
            or (slots is not None and (slots.ndim != 1 or (reqs and (
                positions is None or positions.shape != slots.shape
                or (qsl is None and tokens != reqs)))))
            or (qsl is not None and (not reqs or qsl.shape != (reqs + 1,)))):
        return None
    lib = _lib.load()
    groups = lib.mlr_check_step_groups(reqs, tokens)
    if groups == 0 or (reqs == 0 and tokens == 0):
        return None
    width = stride = 0
    if tables is not None:
        width = tables.shape[1]
        if width > 1 and tables.stride(1) != 1:
            tables = tables.contiguous()
        stride = tables.stride(0) if reqs > 1 else width
        if stride < width:
            tables = tables.contiguous()
            stride = width
    ctx, qsl, positions, slots, decoding = (
        None if t is None else t.contiguous() for t in (ctx, qsl, positions, slots, decoding))
    # The kernel writes its words straight to pinned host memory, read after
    # the wait that the checks cost anyway: no copy behind the kernel. The
    # buffer is this call's own until the wait has ended.
    out = torch.empty(groups + (3 * reqs + 1 if detail else 0), dtype=torch.long,
                      device="cpu", pin_memory=True)  # whatever the default device is

    def ptr(t):
        return None if t is None else t.data_ptr()

    with _lib.on(device):
        status = lib.mlr_check_step_wait(
            ptr(tables), stride, width, ptr(ctx), reqs, ptr(qsl), ptr(positions), ptr(slots),
            tokens, ptr(decoding), block_size, num_blocks, max_query_len, detail,
            out.data_ptr(), out.numel(), _lib.stream_handle(device))
    _lib.check(status, "mlr_check_step_wait")
    host = out.tolist()
    flags = 0
    for word in host[:groups]:
        flags |= word
    if not detail:
        return flags
    host = host[groups:]
    return flags, host[:reqs + 1], host[reqs + 1:2 * reqs + 1], host[2 * reqs + 1:]
