"""Hit lists as the binding returns them, around the hits that come with the
count: complete, in (index, query) order, whoever owns the buffers and on
whichever stream."""
import numpy as np
import pytest

from yume_pdq import synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 1022, 1023, 1024, 1025, 5000])
def test_lists_of_every_length(gpu, dev, n):
    import torch
    q = synthetic.random_db(3, seed=1)
    rows = synthetic.random_db(n + 40, seed=2)
    at = np.sort(np.random.default_rng(3).permutation(n + 40)[:n])
    rows[at] = q[1]
    d, dq = torch.from_numpy(rows).to(dev), torch.from_numpy(q).to(dev)
    want = np.zeros(n, gpu.HIT_DTYPE)
    want["query"], want["index"] = 1, at
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for kw in ({}, {"stream": side}, {"capacity": max(n, 1)}):
        total, hits = gpu.match(d, dq, 20, **kw)
        assert total == n and np.array_equal(hits, want), kw
    own = torch.empty((n + 3, 16), dtype=torch.uint8, device=dev)
    count = torch.full((1,), 77, dtype=torch.int64, device=dev)
    for hits_given, count_given in ((own, None), (None, count), (own, count)):
        total, hits = gpu.match(d, dq, 20, hits=hits_given, count=count_given)
        assert total == n and np.array_equal(hits, want)
    # appended to a list that is there: every hit twice, past the buffer counted only
    total, hits = gpu.match(d, dq, 20, hits=own, count=count, append=True)
    assert total == 2 * n and len(hits) == min(2 * n, n + 3)
    assert np.array_equal(hits, np.sort(hits, order=("index", "query")))
    assert np.array_equal(np.unique(hits), want)
    s = gpu.Shards()
    try:
        s.add(rows[:7])
        s.add(rows[7:])
        total, hits = s.match(dq, 20)
        assert total == n and np.array_equal(hits, want)
        total, hits = s.match(dq[:0], 20)
        assert total == 0 and len(hits) == 0
    finally:
        s.close()


@pytest.mark.parametrize("n", [1, 2, 5, 300])
def test_hash_launch_clears_the_count(gpu, dev, n):
    """The counter of a hash-and-match batch starts from garbage, in every hash
    layout and on repeated runs, with rows and without."""
    import torch
    planes = torch.from_numpy(synthetic.images_u8(8)).to(dev).repeat((n + 7) // 8, 1, 1)[:n].contiguous()
    h = gpu.hash_batch(planes)[0].reshape(-1, 32)
    rows = torch.cat([h[:5], torch.from_numpy(synthetic.random_db(100, seed=3)).to(dev)])
    want, want_hits = gpu.match(rows, h, 10)
    hm = gpu.HashMatch(planes, rows, 10)
    empty = gpu.HashMatch(planes, rows[:0], 10)
    for _ in range(3):
        hm.count.fill_(77)
        empty.count.fill_(77)
        assert hm.run() == want > 0 and np.array_equal(hm.results()[1], want_hits)
        assert empty.run() == 0 and int(empty.count) == 0
    s = gpu.Shards()
    s.add(rows)
    b = gpu.Batcher(s, 300, threshold=10)
    try:
        for use_graph in (True, False, True):
            b.count.fill_(77)
            torch.cuda.synchronize()
            _, _, _, total, hits = b.run(planes, use_graph=use_graph)
            assert total == want and np.array_equal(hits, want_hits)
    finally:
        b.close()
        s.close()


def test_batches_enqueued_without_waiting(gpu, dev):
    """Batches of different sizes enqueued one behind the other, with the shard
    set replaced in between (its graphs are captured again): each has its own
    size and count."""
    import torch
    planes = torch.from_numpy(synthetic.images_u8(64)).to(dev)
    h = gpu.hash_batch(planes)[0].reshape(-1, 32)
    rows = torch.cat([h[::3], torch.from_numpy(synthetic.random_db(1000, seed=4)).to(dev)])
    sizes = [1, 64, 7, 2, 33, 64, 5, 1, 16, 50]
    want = [gpu.match(rows, h[:8 * n], 20)[0] for n in sizes]
    s = gpu.Shards()
    s.add(rows)
    b = gpu.Batcher(s, 64, threshold=20)
    try:
        for turn in range(3):
            got = []
            for n in sizes:
                b.run(planes[:n], sync=False)
                with torch.cuda.stream(b.stream):
                    got.append(b.count.clone())
            if turn == 1:  # a shard without a near row: the counts stay, the graphs do not
                s.add(torch.zeros((9, 32), dtype=torch.uint8, device=dev))
            b.stream.synchronize()
            assert [int(c) for c in got] == want, turn
    finally:
        b.close()
        s.close()
