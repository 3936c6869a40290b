"""Host side of dynamiq_pipeline.SinglePassBuckets on the CPU, over a native module that notes what it is given: who keeps
which memory, in which order launches are enqueued."""
import gc
import threading
import time
import weakref

import pytest
import torch

from dynamiq_sigcomm_artifact_amd import capi
from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets


class _Host(object):
    """stands in for the `_host` module: keeps weak references only, as the launches of a recorded graph do"""

    def __init__(self):
        self.launches = []
        outer = self

        class Buckets(object):
            def __init__(self, strategy, seed, step, u, hist, counts):
                self.recorded = False
                self.counts = counts
                self.stats = self.spare = None

            def scratch(self, stats, spare):
                self.stats, self.spare = stats, spare

            def join(self):
                pass

            def begin_step(self):
                pass

        class Batch(object):
            def __init__(self, buckets, pairs, steps, rows):
                slots, spare = buckets.counts.shape[0], buckets.spare.shape[0]
                assert sum((x.numel() + 255) // 256 for x, _ in pairs) <= buckets.stats.shape[0]
                assert all(0 <= r < slots + spare for r in rows) and len(set(rows)) == len(rows)
                self.seen = [(x.data_ptr(), o.data_ptr(), x.numel()) for x, o in pairs]
                self.rows, self.steps = list(rows), list(steps)

            def matches(self, pairs):
                return [(x.data_ptr(), o.data_ptr(), x.numel()) for x, o in pairs] == self.seen

            def launch(self, buckets):
                outer.launches.append((self, weakref.ref(buckets.stats), weakref.ref(buckets.spare)))

        self.Buckets, self.Batch = Buckets, Batch


@pytest.fixture
def host(monkeypatch):
    h = _Host()
    monkeypatch.setattr(capi, "host", lambda: h)
    return h


def _pairs(*sizes):
    return [(torch.zeros(n), torch.zeros(n)) for n in sizes]


@pytest.mark.parametrize("streams", [1, 3])
def test_scratch_of_a_recorded_launch_lives_as_long_as_the_object(host, streams):
    """a recorded launch writes statistics and counts at every replay: when a larger bucket or a longer list replaces the scratch,
    the old one stays; all that is kept together is no more than the present one"""
    pipe = SinglePassBuckets("cpu", streams=streams)
    small, grown = _pairs(256 * 8, 256 * 3 + 1), _pairs(256 * 9, 256, 256 * 2, 255, 256)
    pipe._buckets.recorded = True                  # as the native object has it from the first recording on
    pipe.run_all(small)
    for pairs in (grown, _pairs(256 * 500), _pairs(*([256] * 40))):
        pipe.run_all(pairs)
    gc.collect()
    assert all(stats() is not None and spare() is not None for _, stats, spare in host.launches)
    assert len({stats().data_ptr() for _, stats, _ in host.launches}) >= 2
    assert sum(s.numel() for s, _ in pipe._replaced) <= pipe._scratch[0].numel()


def test_scratch_without_recordings_is_given_back(host):
    pipe = SinglePassBuckets("cpu")
    pipe.run_all(_pairs(256 * 8))
    pipe.run_all(_pairs(256 * 800))
    gc.collect()
    assert [stats() is None for _, stats, _ in host.launches] == [True, False]


def test_counts_of_a_slot_stay_where_they_are(host):
    """a slot's counts are those of its last bucket, in a row that never moves: a replay after the scratch has grown writes where
    counts() looks"""
    pipe = SinglePassBuckets("cpu", streams=2)
    pairs = _pairs(256, 512, 768)
    pipe.run_all(pairs)
    batch = host.launches[-1][0]
    assert batch.rows[1:] == [1, 0] and batch.rows[0] >= 2          # buckets 0 and 2 share slot 0
    before = [pipe.counts(k).data_ptr() for k in range(2)]
    pipe.run_all(_pairs(*([256 * 300] * 9)))
    assert [pipe.counts(k).data_ptr() for k in range(2)] == before
    assert pipe.run(*pairs[1]) == 1 and host.launches[-1][0].rows == [1]


def test_threads_take_turns(host):
    """a launch gives up the interpreter's lock in the middle: no other call of the object may come in between, and no scratch be
    replaced under a launch that was laid out over it"""
    pipe = SinglePassBuckets("cpu")
    inside, met = [], []

    def alone(body):
        def call(*args):
            inside.append(1)
            if len(inside) > 1:
                met.append(1)
            time.sleep(0.002)
            try:
                return body(*args)
            finally:
                inside.pop()
        return call

    launch = host.Batch.launch

    def over_its_scratch(batch, buckets):
        stats = buckets.stats
        time.sleep(0.002)
        assert buckets.stats is stats
        launch(batch, buckets)

    host.Batch.launch = alone(over_its_scratch)
    pipe._buckets.begin_step = alone(pipe._buckets.begin_step)
    lists = [_pairs(256 * (8 + 300 * k), 256) for k in range(4)]
    failed = []

    def work(k):
        try:
            for _ in range(5):
                pipe.begin_step()
                pipe.run_all(lists[k])
                pipe.run(*lists[k][0])
                pipe.set_u(6.0)
        except Exception as exc:      # noqa: BLE001 (shown by the assertion below)
            failed.append(exc)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(lists))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failed and not met and len(host.launches) == 40
