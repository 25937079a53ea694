"""How steps are filled up to sizes that run well: the rule for rows, and the entry that stands
for a request that does not exist (host logic, no GPU)."""

from types import SimpleNamespace

import pytest

from from_scratch_inference_engine_amd.engine.context import HostBatch, filler_entry, padded_tokens
from from_scratch_inference_engine_amd.engine.graphs import padded_rows


def test_rows_of_a_step_that_is_not_a_decode_step():
    assert [padded_tokens(n) for n in (1, 2, 64)] == [1, 2, 64]
    assert [padded_tokens(n) for n in (65, 100, 128)] == [128, 128, 128]
    # the next multiple of 256 where that adds at most a fifth, or 64 rows
    assert [padded_tokens(n) for n in (129, 192, 200, 300, 448, 777, 1000, 1088, 2048, 3000)] == \
        [129, 256, 256, 300, 512, 777, 1024, 1280, 2048, 3072]
    for n in range(1, 5000):
        up = padded_tokens(n)
        assert n <= up < n + 256 and (up == n or up % 128 == 0) and padded_tokens(up) == up


def test_rows_of_a_decode_graph():
    assert [padded_rows(n) for n in range(1, 10)] == [1, 2, 4, 4, 8, 8, 8, 8, 16]
    for n in range(1, 300):
        up = padded_rows(n)
        assert n <= up <= max(2 * n, n + 31) and padded_rows(up) == up


def test_the_filler_reads_and_writes_spare_places_only():
    # two groups of layers; a page of the second holds 16 positions (a need with a geometry of its own)
    storage = SimpleNamespace(spare_slot=5, spare_pages=[40, 17], tokens_per_page=[8, 16])
    e = filler_entry(storage, 37)
    assert len(e.tokens) == 37 and set(e.tokens) == {0} and tuple(e.want) == ()
    assert e.cache.length == 0 and e.cache.slot == 5
    assert e.cache.tables == [[40] * 5, [17] * 3]          # every page of its table is the spare one
    host = HostBatch([e], page_size=8)
    assert host.n_tokens == 37 and host.positions.tolist() == list(range(37)) and host.want_rows.size == 0


@pytest.mark.parametrize("was_on", [True, False])
def test_the_collector_is_off_until_the_last_capture_ends(was_on):
    import gc

    from from_scratch_inference_engine_amd.engine.graphs import _collector_off

    before = gc.isenabled()
    (gc.enable if was_on else gc.disable)()
    try:
        with _collector_off:
            with pytest.raises(RuntimeError):
                with _collector_off:
                    raise RuntimeError("a capture that fails")
            assert not gc.isenabled()
        assert gc.isenabled() == was_on
    finally:
        (gc.enable if before else gc.disable)()


def test_graphs_go_with_the_weight_copies_that_they_read():
    """A second runner whose cache does not fit beside the second copies of the weights takes their memory; what the first runner has captured
    reads them, so none of it may be replayed again."""
    from from_scratch_inference_engine_amd.engine.graphs import DecodeGraphs

    class Runner:
        model = SimpleNamespace(spec=SimpleNamespace(all_parts=lambda: []), planners=[], copies_dropped=0)
        storage = SimpleNamespace(spare_slot=0, spare_pages=[], tokens_per_page=[])

    class Captured:
        def replay(self):
            raise AssertionError("replayed")

    runner = Runner()
    graphs = DecodeGraphs(runner, capture_after=3)
    graphs._graphs[(1, ("pages", 32))] = (Captured(), None, None, None)
    runner.model.copies_dropped += 1
    entry = SimpleNamespace(tokens=(1,), want=(0,), cache=SimpleNamespace(tables=[], length=3, slot=0))
    assert graphs.step([entry], {"pages": 32}) is None and not graphs._graphs
    graphs._graphs[(1, ("pages", 32))] = "a new one"
    graphs.step([entry] * 2, {"pages": 32})
    assert graphs._graphs  # (once for each time that they go)
