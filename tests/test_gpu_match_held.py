"""The matrix-core matcher's held-rows layout at its edges: rows around a wave's
192 and 128 and a block's part, queries around its tiles, pairs and votes of
eight tiles, 64 tiles and several chunks, thresholds around the change from two
to three products per accumulator, the lines of its rule, dense hits."""
import numpy as np
import pytest

from yume_pdq import synthetic

pytestmark = pytest.mark.gpu


def triples(hits):
    return np.stack([hits["query"], hits["index"], hits["distance"]], 1).astype(np.int64)


def planted(n_rows, queries, seed):
    """Random rows; up to 300 of them near-duplicates of random queries, the
    first and the last row and queries among them."""
    db = synthetic.random_db(n_rows, seed=seed)
    rng = np.random.default_rng(seed)
    rows = np.unique(np.concatenate([[0, n_rows - 1], rng.integers(0, n_rows, 298)]))
    which = rng.integers(0, len(queries), len(rows))
    which[0], which[-1] = 0, len(queries) - 1
    for r, w in zip(rows, which):
        db[r] = synthetic.flip_bits(queries[w], int(rng.integers(0, 70)), rng)
    return db


@pytest.mark.parametrize("n_rows", [1, 127, 128, 129, 191, 192, 193, 385, 1535, 1537, 12289, 50001])
@pytest.mark.parametrize("nq", [65, 128, 129, 144, 161, 257, 1008, 1024, 1025, 1153, 2100])
def test_edges(gpu, oracle, dev, n_rows, nq):
    import torch
    queries = synthetic.random_db(nq, seed=nq)
    db = planted(n_rows, queries, 2000 + n_rows)
    d, q = torch.from_numpy(db).to(dev), torch.from_numpy(queries).to(dev)
    plane = gpu.build_prefix_plane(d)
    for threshold in (27, 28, 63):
        n, want = oracle.match_all_mt(db, queries, threshold)
        for p in (None, plane):
            total, hits = gpu.match(d, q, threshold, plane=p, index_base=7)
            where = f"{n_rows} x {nq}, threshold {threshold}, plane {p is not None}"
            assert total == n, where
            got = triples(hits)
            got[:, 1] -= 7
            assert np.array_equal(got, want), where


@pytest.mark.parametrize("n_rows,nq", [(300_000, 200), (699_999, 193), (700_001, 193), (400_000, 1100)])
def test_many_rows(gpu, dev, n_rows, nq):
    """Several row groups per wave: the vector-ALU matcher's set."""
    import torch
    g = torch.Generator(device=dev).manual_seed(n_rows)
    db = torch.randint(-(1 << 63), (1 << 63) - 1, (n_rows, 4), generator=g, device=dev).view(torch.uint8)
    db = db.reshape(n_rows, 32)
    q = torch.from_numpy(synthetic.random_db(nq, seed=12)).to(dev)
    at = torch.randperm(n_rows, generator=g, device=dev)[:3000]
    db[at] = q[torch.arange(3000, device=dev) % nq] ^ (torch.randint(0, 256, (3000, 1), generator=g, device=dev)
                                                       .to(torch.uint8) & 17)
    db[0], db[n_rows - 1] = q[0], q[nq - 1]
    plane = gpu.build_prefix_plane(db)
    for threshold in (20, 31, 40):
        n0, h0 = gpu.match(db, q, threshold, path="valu")
        for p in (None, plane):
            n1, h1 = gpu.match(db, q, threshold, plane=p)
            assert n0 == n1 > 0 and np.array_equal(triples(h0), triples(h1)), (threshold, p is not None)


def test_every_pair_a_hit(gpu, dev):
    """More hits than a block's list, into a buffer that holds them and one
    that does not (the count stays exact)."""
    import torch
    row = synthetic.random_db(1, seed=5)
    d = torch.from_numpy(np.repeat(row, 500, 0)).to(dev)
    q = torch.from_numpy(np.repeat(row, 200, 0)).to(dev)
    total, hits = gpu.match(d, q, 31, capacity=500 * 200)
    assert total == 500 * 200 and (hits["distance"] == 0).all()
    assert np.array_equal(hits["index"], np.repeat(np.arange(500), 200))
    assert np.array_equal(hits["query"], np.tile(np.arange(200), 500))
    total, hits = gpu.match(d, q, 31, capacity=1000)
    assert total == 500 * 200 and len(hits) == 1000
