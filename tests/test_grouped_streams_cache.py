"""The kept grouped streams (fused_factored.grouped_streams): what stays, what
goes and what a device's bound counts; on the CPU, where the share of the
device's memory is none."""

import pytest
import torch

import problems
from gm_attention_amd.nn import fused_factored


@pytest.fixture(autouse=True)
def empty(monkeypatch):
    monkeypatch.setattr(fused_factored, "_STREAMS", type(fused_factored._STREAMS)())


def _edges(n, nlat=6):
    one = problems.discretization(nlat, 2 * nlat).edge_geometry.to("cpu", torch.float32)
    return [one.tile(2 + i % 3, n_sources=2 * nlat * nlat) for i in range(n)]


def _streams(edges, phases=False):
    order = fused_factored.groups_for(edges, edges.source_index)[0]
    return fused_factored.grouped_streams(edges, order, 0.5, 5, 3, torch.float32, phases)


def _kept():
    return [s for _, s in fused_factored._STREAMS.values()]


def test_no_more_is_kept_than_eight_sets_with_phase_rows_take():
    sets = _edges(40)
    for e in sets:
        s = _streams(e)
        assert s.phase_g is None and s.bytes(phases=True) == s.bytes() + 64 * e.n_edges
        kept = _kept()
        assert kept[-1] is s
        assert sum(k.bytes() for k in kept) <= sum(k.bytes(phases=True) for k in kept[-8:])
    assert fused_factored.STREAMS_SHARE <= 1 / 128  # beyond that: of the device's memory
    assert len(_kept()) > 16  # 36 bytes an edge against 100
    assert _streams(sets[-1]) is _kept()[-1] and _streams(sets[-8]) is _kept()[-1]  # used again: the last to go
    fused_factored.release_streams()
    assert not _kept()


def test_sets_with_phase_rows_are_the_last_eight():
    sets = _edges(12)
    made = [_streams(e, phases=True) for e in sets]
    assert all(a is b for a, b in zip(_kept(), made[-8:], strict=False)) and len(_kept()) <= 9


def test_streams_go_with_their_edge_set():
    sets = _edges(3)
    for e in sets:
        _streams(e)
    assert len(_kept()) == 3
    del sets[0], e
    _streams(sets[0], phases=True)
    assert len(_kept()) == 3  # two sets, one of them with and without phase rows


def test_one_devices_bound_drops_nothing_of_another():
    class Elsewhere:
        """Streams of another device that fit its bound, as far as the bound looks at them."""

        inv = torch.empty(0, device="meta")

        def bytes(self, phases=False):
            return 0

    owner = torch.zeros(1)
    fused_factored._STREAMS["other"] = (lambda: owner, Elsewhere())
    sets = _edges(40)
    for e in sets:
        _streams(e)
    assert len(_kept()) < len(sets) and next(iter(fused_factored._STREAMS)) == "other"


def _recorded(monkeypatch):
    """What is done about other streams, in order, with what the caches hold meanwhile."""
    native, seen = fused_factored._native, []
    monkeypatch.setattr(fused_factored, "_GROUPS", type(fused_factored._GROUPS)())
    monkeypatch.setattr(native, "_GROUPS", {})
    monkeypatch.setattr(native, "_GROUPED_TABLES", {})
    caches = lambda: (len(fused_factored._GROUPS), len(fused_factored._STREAMS),  # noqa: E731
                      len(native._GROUPS), len(native._GROUPED_TABLES))
    monkeypatch.setattr(native, "complete", lambda device: seen.append(("complete", caches())))
    made, found = native.Made.__init__, native.Made.found
    monkeypatch.setattr(native.Made, "__init__", lambda self, *t: (seen.append(("made", caches())), made(self, *t))[1])
    monkeypatch.setattr(native.Made, "found", lambda self: (seen.append(("found", caches())), found(self))[1])
    return seen


def test_groups_are_complete_and_streams_marked_before_they_are_kept(monkeypatch):
    seen = _recorded(monkeypatch)
    edges, = _edges(1)
    _streams(edges)
    assert seen == [("complete", (0, 0, 0, 0)), ("made", (1, 0, 0, 0))]
    _streams(edges)
    assert seen[2:] == [("found", (1, 1, 0, 0))]


def test_the_transposed_grouping_is_complete_and_its_tables_marked_before_they_are_kept(monkeypatch):
    seen = _recorded(monkeypatch)
    native = fused_factored._native
    edges, = _edges(1)
    source, transport = edges.source_index.contiguous(), torch.view_as_real(edges.transport_phases).contiguous()
    target_s, inv, _ = native.source_grouped_tables(source, edges.row_ptr, transport)
    assert seen == [("complete", (0, 0, 0, 0)), ("made", (0, 0, 1, 0))]
    order = torch.argsort(source, stable=True)
    assert torch.equal(target_s.long(), edges.target_index[order])
    assert torch.equal(order[inv.long()], torch.arange(order.numel()))
    native.source_grouped_tables(source, edges.row_ptr, transport)
    assert seen[2:] == [("found", (0, 0, 1, 1))]


@pytest.mark.gpu
def test_streams_made_behind_a_busy_stream_are_waited_for_by_another(cuda):
    native = fused_factored._native
    edges = problems.discretization(9, 18).edge_geometry.to(cuda, torch.float32)
    source, transport = edges.source_index.contiguous(), torch.view_as_real(edges.transport_phases).contiguous()
    order = torch.argsort(source, stable=True)
    native.source_major(source, edges.row_ptr)
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(first):
        fused_factored.groups_for(edges, edges.source_index)
        torch.cuda._sleep(100_000_000)  # some tens of milliseconds ahead of the tables
        got = _streams(edges, phases=True)
        tables = native.source_grouped_tables(source, edges.row_ptr, transport)
    with torch.cuda.stream(second):
        assert _streams(edges, phases=True) is got
        read = got.target_g.clone(), got.perm.clone()
        again = native.source_grouped_tables(source, edges.row_ptr, transport)
        assert again is tables
        read += tuple(t.clone() for t in again)
        second.synchronize()
        assert first.query()  # the reads came after what made them
    assert torch.equal(read[1], order) and torch.equal(read[0], edges.target_index[order])
    assert torch.equal(read[2].long(), edges.target_index[order]) and torch.equal(read[4], transport[order])


def test_the_low_passes_transpose_is_complete_before_it_is_kept(monkeypatch):
    from gm_attention_amd.nn import segformer

    edges, = _edges(1)
    kept = []
    monkeypatch.setattr(fused_factored._native, "complete",
                        lambda device: kept.append([k for k in edges.__dict__ if "_low_pass_transpose" in k]))
    n = edges.row_ptr.shape[0] - 1
    src_ptr, order, target = segformer._transpose(edges, n)
    assert kept == [[]] and segformer._transpose(edges, n)[0] is src_ptr and len(kept) == 1
    assert torch.equal(target, edges.target_index[order]) and int(src_ptr[-1]) == edges.n_edges
