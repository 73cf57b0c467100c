"""Plans built on the device (wmx_plan_count / wmx_plan_fill) against the host
builders on CPU copies of the same tensors, entry for entry: cyclic document
metadata at strides, residues, dummies, documents and lengths around the
builders' chunks (1,024 segments and 4,096 queries or keys of a row a round, 256
units of a list), metadata that is not run-structured, and packed schedules with
padding, short histories and the dummy. The host builders are pinned by the
oracle on the CPU (tests/test_cyclic_packing.py, tests/test_host.py)."""

import importlib

import numpy as np
import pytest
import torch

import bench
from white_matter_amd import prepare_cyclic_attention_metadata, prepare_feedback_metadata, prepare_strict_causal_metadata
from white_matter_amd import _plans

cyclic = importlib.import_module("white_matter_amd.cyclic_attention")
strict = importlib.import_module("white_matter_amd.strict_causal_attention")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _same(device, host, what):
    assert len(device) == len(host), what
    for n, (d, h) in enumerate(zip(device, host)):
        assert d.dtype == h.dtype and d.shape == h.shape and torch.equal(d.cpu(), h), f"{what}: output {n}"


def _compare_cyclic(meta, q_len, k_len, stride, offset, what, planned=True):
    """The status, and whether the device planned it (which `planned` asks for)."""
    meta = [t.to(DEV, torch.int32).contiguous() for t in meta]
    host = cyclic._cyclic_schedule(*(t.cpu() for t in meta), q_len, k_len, stride, offset)
    built = _plans.cyclic_plan(meta, q_len, k_len, stride, offset, strict._key_tile(None, stride), strict._FUSED_ROWS)
    assert built is not None or not planned, f"{what}: the host's builder planned it"
    _same(cyclic._cyclic_schedule(*meta, q_len, k_len, stride, offset), host, what)
    return int(host[0][0]), built is not None


@pytest.mark.parametrize("dummy", [False, True])
@pytest.mark.parametrize(("length", "mean", "stride"), [(40, 6, 3), (333, 50, 8), (1024, 200, 2), (2100, 300, 1), (9, 30, 4)])
def test_cyclic_plans_match_the_host_builder(length, mean, stride, dummy):
    docs = bench.geometric_documents(3, length, seed=length + stride, mean=mean, lo=1, hi=length).to(DEV)
    docs[1] = 0  # a row of one document
    groups = [torch.arange(r, length, stride, device=DEV) for r in range(stride)]
    metas = prepare_feedback_metadata(docs, groups, length + int(dummy), use_dummy_token=dummy)
    for r, meta in enumerate(metas):
        offset = r if dummy else r - 1
        status, _ = _compare_cyclic(meta, groups[r].numel(), length + int(dummy), stride, offset, f"residue {r}")
        assert status in (1, 2)


@pytest.mark.parametrize("dummy", [False, True])
@pytest.mark.parametrize(
    ("length", "mean", "stride"),
    [
        (4096, 700, 1),  # one chunk of queries and keys, and (4097) one entry of the next
        (4097, 700, 1),
        (9000, 5000, 1),  # a document across chunks
        (9000, 4, 1),  # over 1,024 segments in a row
        (9001, 400, 2),
        (16500, 40, 4),  # segments past 1,024 in all, keys past four chunks
    ],
)
def test_cyclic_plans_past_a_chunk(length, mean, stride, dummy):
    """What the scans carry from chunk to chunk: places, segments, coverage and
    runs, with queries and keys of no segment on either side of a boundary."""
    docs = bench.geometric_documents(3, length, seed=length + mean, mean=mean, lo=1, hi=length)
    docs[1] = 0
    docs[2, 4090:4100] = torch.arange(4090, 4100)[: docs[2, 4090:4100].numel()] + length  # single tokens around the boundary
    docs = docs.to(DEV)
    groups = [torch.arange(r, length, stride, device=DEV) for r in range(stride)]
    metas = prepare_feedback_metadata(docs, groups, length + int(dummy), use_dummy_token=dummy)
    for r in {0, stride - 1}:
        q_len, k_len, offset = groups[r].numel(), length + int(dummy), r if dummy else r - 1
        what = f"residue {r}"
        assert _compare_cyclic(metas[r], q_len, k_len, stride, offset, what)[0] == 2
        # fewer queries than keys: the keys past the last one's document lie in no segment
        few = q_len // 3
        meta = [t[:, :few] if n in (0, 2) else t for n, t in enumerate(metas[r])]
        meta[3] = meta[3].clamp_max(few)
        meta[3][meta[1] < 0] = few
        assert _compare_cyclic(meta, few, k_len, stride, offset, f"{what}, a third of the queries")[0] == 2


def test_plans_of_other_metadata_match_the_host_builder():
    """Shorter key ranges, two dummies, repeated labels and random metadata:
    the same plan, or the same refusal."""
    rng = np.random.default_rng(5)
    seen = set()
    for trial in range(60):
        batch, q_len, stride = int(rng.integers(1, 4)), int(rng.integers(1, 40)), int(rng.integers(1, 4))
        k_len = stride * (q_len - 1) + 1 + int(rng.integers(0, 20))
        ids = np.sort(rng.integers(0, 5, (batch, k_len)), 1)
        kind = trial % 4
        keys = torch.from_numpy(ids)
        if kind == 0:
            keys[:, : int(rng.integers(0, 3))] = -1
        queries = keys[:, torch.arange(q_len) * stride].clamp_min(0)
        qstart = torch.searchsorted(keys, queries, right=False)
        kqend = torch.searchsorted(queries, keys, right=True)
        kqend[keys < 0] = q_len
        if kind == 1:  # a label that returns later in the row
            keys[:, k_len // 2 :] = keys[:, k_len // 2 :] % 2
        if kind == 2:
            qstart = qstart + torch.from_numpy(rng.integers(-2, 3, qstart.shape))
        if kind == 3:
            kqend = torch.from_numpy(rng.integers(0, q_len + 1, kqend.shape))
        offset = int(rng.integers(-1, stride))
        meta = (queries, keys, qstart, kqend)
        seen.add(_compare_cyclic(meta, q_len, k_len, stride, offset, f"trial {trial}", planned=False))
    assert seen >= {(0, True), (2, True)}


def _compare_packed(meta, batch, length, slots, what, planned=True):
    given = (meta.query_indices, meta.key_indices, meta.cu_queries, meta.cu_keys)
    shape = (meta.max_queries, meta.max_keys, batch, length, slots, 4, 2)
    host = strict._packed_plan(*(t.cpu() for t in given), *shape)
    assert _plans.packed_plan(given, batch, length, slots, strict._key_tile(None)) is not None or not planned, what
    device = strict._packed_plan(*given, *shape)
    for n in (0, *range(1, 11)):
        if host[n].numel() or device[n].numel():
            _same([device[n]], [host[n]], f"{what}: output {n}")
    return host


@pytest.mark.parametrize("dummy", [False, True])
@pytest.mark.parametrize(
    ("length", "mean"),
    [(17, 4), (300, 40), (1025, 90), (2500, 600), (4097, 300), (9000, 4), (9000, 3000)],
)
def test_packed_plans_match_the_host_builder(length, mean, dummy):
    docs = bench.geometric_documents(3, length, seed=length, mean=mean, lo=1, hi=length).to(DEV)
    docs[1, length // 3 : length // 2] = -1  # padding inside a row
    docs[2, -3:] = -1
    meta = prepare_strict_causal_metadata(docs, length, use_dummy_token=dummy)
    host = _compare_packed(meta, 3, length, length + int(dummy), "documents")
    assert int(host[0][0]) >= meta.cu_queries.numel() - 1
    # queries behind a cached prefix: key rows repeat across segments (the host plans those), or sit in a wider pool
    prefix = length // 2
    late = prepare_strict_causal_metadata(
        docs.abs(), length - prefix, query_start=prefix, use_dummy_token=dummy,
        kv_lengths=torch.tensor([prefix, length, prefix + 3], device=DEV),
    )
    _compare_packed(late.with_key_extent(length + 40), 3, length - prefix, length + 40, "cached prefix", planned=False)


def test_plans_take_the_device_path():
    """The benchmark's forms are planned on the device, not by the host builders."""
    docs = bench.geometric_documents(2, 512, seed=1).to(DEV)
    meta = prepare_strict_causal_metadata(docs, 512, use_dummy_token=True)
    given = (meta.query_indices, meta.key_indices, meta.cu_queries, meta.cu_keys)
    assert _plans.packed_plan(given, 2, 512, 513, 128) is not None
    ids = torch.cat((torch.full((2, 1), -1, device=DEV), docs), 1)
    cyc = prepare_cyclic_attention_metadata(docs[:, ::4].contiguous(), ids)
    assert _plans.cyclic_plan(tuple(cyc), 128, 513, 4, 0, 64, 96)[0][0] == 2


@torch.no_grad()
def test_schedules_without_keys_or_queries():
    """Segments without keys give zeros, and a schedule without queries or keys
    is planned as on the host (an empty tensor's address reads as missing)."""
    ints = lambda *v: torch.tensor(v, device=DEV, dtype=torch.int32)  # noqa: E731
    none = torch.empty(0, device=DEV, dtype=torch.int64)
    rows = torch.tensor([0, 1, 2, 5, 6], device=DEV)
    metadata = strict.StrictCausalMetadata(rows, none, ints(0, 3, 5), ints(0, 0, 0), 4, 6, 6)
    _compare_packed(metadata, 2, 4, 6, "no keys", planned=False)
    no_queries = strict.StrictCausalMetadata(none, torch.arange(3, device=DEV), ints(0, 0), ints(0, 3), 4, 6, 6)
    _compare_packed(no_queries, 2, 4, 6, "no queries", planned=False)
    _compare_packed(strict.StrictCausalMetadata(none, none, ints(0, 0), ints(0, 0), 4, 6, 6), 2, 4, 6, "neither", planned=False)
    q, k, v = (torch.randn(2, 2, n, 64, device=DEV).bfloat16() for n in (4, 6, 6))
    assert not strict.strict_causal_attention(q, k, v, metadata=metadata).any()
