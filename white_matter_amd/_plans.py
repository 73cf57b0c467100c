"""Plans of packed attention calls built on the device (wmx_plan_count,
wmx_plan_fill): the schedules, work lists and dS layouts that
`_cyclic_schedule` and `_packed_plan` otherwise build from torch operations
and host lists, entry for entry the same. One read of the counts sizes the
outputs; a second synchronisation ends the build, so that a cached plan can be
used from any stream.

Both builders return None for what the kernels do not plan (see
WMX_PLAN_GENERAL in wmx_attn.h); the host builders then decide, raise or plan
it.
"""

from __future__ import annotations

import torch

from . import _native

_MAX_SEGMENTS = (1 << 20) - 1  # a sort key's segment and tile fields (csrc/plan.hip)
_MAX_TILES = (1 << 15) - 1
_MAX_COUNT = (1 << 21) - 1  # rows, keys and units that its scans count in one word


class _Counts:
    """The counts of a plan over all rows."""

    def __init__(self, counts: torch.Tensor) -> None:
        host = counts.cpu().numpy()
        (
            self.queries, self.segments, self.keys, self.idle_queries, self.query_runs, self.idle_keys, self.key_runs, _, _,
            self.q_units, self.k_units, self.f_units, self.bq_units, self.bk_units, self.ds_elements, _, self.dummies,
        ) = host.sum(0).tolist()
        self.max_queries, self.max_keys = host[:, 7].max().item(), host[:, 8].max().item()
        flags = int(host[:, 15].max())  # 1, 2 or 3 where a row has any
        self.refused = bool((host[:, 15] & _native.PLAN_REFUSED).any()) if flags else False
        self.general = bool((host[:, 15] & _native.PLAN_GENERAL).any()) if flags else False
        self.rows = host

    def fits(self, batch: int, q_len: int, k_len: int, key_tile: int, total_segments: int) -> bool:
        """The plan stays within int32 and the sort keys' fields."""
        return (
            total_segments <= _MAX_SEGMENTS
            and -(-self.max_queries // 128) <= _MAX_TILES
            and -(-self.max_keys // key_tile) <= _MAX_TILES
            and max(self.q_units, self.k_units) <= _MAX_COUNT
            and max(self.queries + self.idle_queries, self.keys + self.idle_keys, batch * max(q_len, k_len)) < 2**31
        )


def _fill(a: _native.PlanArgs, counts: _Counts, total_segments: int, device: torch.device):
    """Allocates the work lists and runs wmx_plan_fill: (q_units, k_units,
    ds_offsets, f_units, bq_units, bk_units); the last three for fused_rows."""

    def rows(n: int) -> torch.Tensor:
        # an empty list keeps an allocation of its own (empty device tensors
        # share a null address, which reads as aliasing)
        return torch.empty(max(n, 1), _native.UNIT_FIELDS, device=device, dtype=torch.int32)[:n]

    a.total_segments = total_segments
    a.num_q_units, a.num_k_units, a.num_f_units = counts.q_units, counts.k_units, counts.f_units
    q_units, k_units = rows(counts.q_units), rows(counts.k_units)
    ds_offsets = torch.empty(total_segments + 1, device=device, dtype=torch.int64)
    a.q_units, a.k_units, a.ds_offsets = q_units.data_ptr(), k_units.data_ptr(), ds_offsets.data_ptr()
    lists = [q_units, k_units, ds_offsets]
    if a.fused_rows:
        fused = [rows(n) for n in (counts.f_units, counts.bq_units, counts.bk_units)]
        # an empty list's pointer is never written through
        a.f_units, a.bq_units, a.bk_units = (t.untyped_storage().data_ptr() for t in fused)
        lists += fused
    units = torch.empty(max(_native.plan_unit_workspace_size(a), 16), device=device, dtype=torch.uint8)
    a.unit_workspace, a.unit_workspace_bytes = units.data_ptr(), units.numel()
    _native.plan_fill(a, device)
    torch.cuda.current_stream(device).synchronize()
    return lists


def cyclic_plan(
    meta: tuple[torch.Tensor, ...], q_len: int, k_len: int, stride: int, offset: int, key_tile: int, fused_rows: int
) -> tuple[tuple[int, ...], list[torch.Tensor]] | None:
    """The plan of int32 contiguous cyclic document metadata on the GPU: the
    facts of `_cyclic_schedule` and its tensors."""
    device = meta[0].device
    batch = meta[0].shape[0]
    if max(q_len, k_len) > _MAX_COUNT or batch * max(q_len, k_len) >= 2**31:
        return None
    a = _native.PlanArgs()
    a.q_seg, a.k_seg, a.q_start, a.k_qend = (t.data_ptr() for t in meta)
    a.batch, a.q_len, a.k_len, a.query_stride, a.query_offset = batch, q_len, k_len, stride, offset
    a.key_tile, a.fused_rows = key_tile, fused_rows
    workspace = torch.empty(_native.plan_workspace_size(a), device=device, dtype=torch.uint8)
    lines = torch.empty(batch, _native.PLAN_COUNTS, device=device, dtype=torch.int64)
    a.workspace, a.workspace_bytes, a.counts = workspace.data_ptr(), workspace.numel(), lines.data_ptr()
    _native.plan_count(a, device)
    c = _Counts(lines)
    dummies = c.rows[:, 16]
    if c.refused or bool((dummies != dummies[0]).any()):
        return (0,), []
    if c.queries == 0:
        return (1,), []
    total = c.segments + c.query_runs + c.key_runs
    if c.general or not c.fits(batch, q_len, k_len, key_tile, total):
        return None
    # the dummy is the one key row that several segments of a row hold
    unique = 2 if dummies[0] and int(c.rows[:, 1].max()) > 1 else 1
    index = [torch.empty(n, device=device, dtype=torch.int64) for n in (c.queries + c.idle_queries, c.keys + c.idle_keys)]
    bounds = [torch.empty(total + 1, device=device, dtype=torch.int32) for _ in range(2)]
    a.out_query_indices, a.out_key_indices = (t.data_ptr() for t in index)
    a.out_cu_queries, a.out_cu_keys = (t.data_ptr() for t in bounds)
    lists = _fill(a, c, total, device)
    # consecutive slots of one row on both sides: all four segment_layout bits
    return (2, total, c.max_queries, c.max_keys, 15, unique, c.ds_elements, key_tile), [*index, *bounds, *lists]


def packed_plan(
    schedule: tuple[torch.Tensor, ...], batch: int, length: int, key_slots: int, key_tile: int
) -> tuple[tuple[int, ...], list[torch.Tensor]] | None:
    """The plan of a packed schedule (int64 query_indices and key_indices,
    int32 cu_queries and cu_keys, contiguous on the GPU): the facts of
    `_packed_plan`, the covering schedule's four tensors (none when it is the
    schedule itself) and the work lists."""
    device = schedule[0].device
    segments = schedule[2].numel() - 1
    if schedule[0].numel() == 0 or schedule[1].numel() == 0:
        return None  # (an empty tensor's address is null, which reads as missing)
    if segments < 1 or segments > _MAX_SEGMENTS or schedule[3].numel() != segments + 1:
        return None
    if max(length, key_slots) > _MAX_COUNT or batch * max(length, key_slots) >= 2**31:
        return None
    a = _native.PlanArgs()
    a.query_indices, a.key_indices, a.cu_queries, a.cu_keys = (t.data_ptr() for t in schedule)
    a.num_queries, a.num_keys, a.num_segments = schedule[0].numel(), schedule[1].numel(), segments
    a.batch, a.q_len, a.k_len, a.query_stride, a.key_tile = batch, length, key_slots, 1, key_tile
    size = _native.plan_workspace_size(a)
    lines_bytes = (batch + 1) * _native.PLAN_COUNTS * 8
    # the seen counters and the counts, cleared together
    cleared = torch.zeros(lines_bytes + size + 16, device=device, dtype=torch.uint8)
    lines = cleared[:lines_bytes].view(torch.int64).view(batch + 1, _native.PLAN_COUNTS)
    at = -(-lines_bytes // 16) * 16
    a.counts, a.workspace, a.workspace_bytes = cleared.data_ptr(), cleared.data_ptr() + at, cleared.numel() - at
    _native.plan_count(a, device)
    c = _Counts(lines)
    total = segments + c.query_runs + c.key_runs
    if c.refused or c.general or max(a.num_queries, a.num_keys) + c.idle_queries + c.idle_keys >= 2**31:
        return None
    if not c.fits(batch, length, key_slots, key_tile, total):
        return None
    cover: list[torch.Tensor] = []
    if total > segments:
        cover = [
            torch.empty(n, device=device, dtype=dtype)
            for n, dtype in (
                (a.num_queries + c.idle_queries, torch.int64), (a.num_keys + c.idle_keys, torch.int64),
                (total + 1, torch.int32), (total + 1, torch.int32),
            )
        ]
        a.out_query_indices, a.out_key_indices, a.out_cu_queries, a.out_cu_keys = (t.data_ptr() for t in cover)
    lists = _fill(a, c, total, device)
    facts = (total, c.max_queries, c.max_keys, 15, 2 if c.dummies else 1, c.ds_elements, int(bool(cover)), key_tile)
    return facts, [*cover, *lists]
