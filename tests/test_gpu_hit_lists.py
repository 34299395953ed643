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
