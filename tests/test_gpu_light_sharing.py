"""Light k = 3 clique roots: the untouched roots of a batch's ranges are given
away, and a launch of nothing else ends when its watchdog expires."""
import numpy as np
import pytest

import dumato_amd as dm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    return dm.Graph.erdos_renyi(60000, 600000, 3)


def test_untouched_roots_of_a_range_are_given_away(graph):
    # fewer ranges of 32 roots than workers
    want = graph.clique_count(3)
    batch = dm.Batch([graph])
    print("case batch ER clique k=3", flush=True)
    res, _ = batch.run([(0, "clique", 3)])
    assert res[0] == want
    assert batch.last_stats()["donations"] > 0


def test_watchdog_is_looked_at(graph):
    # one worker and some thousand batches: no idle worker looks for it
    cfg = dict(blocks=1, waves_per_block=1, vwave=64)
    print("case one worker, k=3", flush=True)
    assert graph.clique_count(3, dm.config(**cfg)) == graph.clique_count(3)
    assert graph.last_stats()["device_ms"] > 0
    print("case one worker, k=3, watchdog", flush=True)
    with pytest.raises(dm.DMError) as e:
        graph.clique_count(3, dm.config(watchdog_s=1e-4, **cfg))
    assert "watchdog" in str(e.value)
    assert graph.clique_count(3, dm.config(watchdog_s=60.0, **cfg)) > 0
