"""The matrix-core matcher's even layout at its edges -- rows around its 64-row
groups, parts and rounds, queries around its tiles and query groups, thresholds
around the change from two to three products per accumulator, hits past a
block's list, shards of every such size -- and the rule that leaves full groups of 64 query tiles over
many rows to the shared-rows layout, with and without room for its records."""
import numpy as np
import pytest

from yume_pdq import synthetic

pytestmark = pytest.mark.gpu


def triples(hits):
    return np.stack([hits["query"], hits["index"], hits["distance"]], 1).astype(np.int64)


def planted(n_rows, queries, seed):
    """Random rows; up to 200 of them near-duplicates of random queries, the
    first and the last row among them."""
    db = synthetic.random_db(n_rows, seed=seed)
    rng = np.random.default_rng(seed)
    rows = np.unique(np.concatenate([[0, n_rows - 1], rng.integers(0, n_rows, 198)]))
    for r in rows:
        db[r] = synthetic.flip_bits(queries[rng.integers(0, len(queries))], int(rng.integers(0, 70)), rng)
    return db


# rows: one, around a group, a round of four groups, a part of 64, and two parts
@pytest.mark.parametrize("n_rows", [1, 63, 64, 65, 255, 257, 4095, 4097, 9000])
# queries: around one tile pair, every width up to sixteen tiles, two and three groups
@pytest.mark.parametrize("nq", [32, 33, 65, 97, 129, 161, 193, 225, 257, 400, 513])
def test_edges(gpu, oracle, dev, n_rows, nq):
    import torch
    queries = synthetic.random_db(nq, seed=nq)
    db = planted(n_rows, queries, 1000 + n_rows)
    d, q = torch.from_numpy(db).to(dev), torch.from_numpy(queries).to(dev)
    plane = gpu.build_prefix_plane(d)
    for threshold in (0, 27, 28, 63):
        n, want = oracle.match_all(db, queries, threshold)
        for p in (None, plane):
            total, hits = gpu.match(d, q, threshold, plane=p)
            where = f"{n_rows} x {nq}, threshold {threshold}, plane {p is not None}"
            assert total == n and np.array_equal(triples(hits), want), where


@pytest.mark.parametrize("nq", [48, 600])
def test_more_hits_than_a_block_lists(gpu, dev, nq):
    """Every pair a hit: 700 rows x nq equal hashes, into a buffer that holds
    them and one that does not (the count stays exact)."""
    import torch
    row = synthetic.random_db(1, seed=5)
    d = torch.from_numpy(np.repeat(row, 700, 0)).to(dev)
    q = torch.from_numpy(np.repeat(row, nq, 0)).to(dev)
    total, hits = gpu.match(d, q, 31, capacity=700 * nq)
    assert total == 700 * nq and (hits["distance"] == 0).all()
    assert np.array_equal(hits["index"], np.repeat(np.arange(700), nq))
    assert np.array_equal(hits["query"], np.tile(np.arange(nq), 700))
    total, hits = gpu.match(d, q, 31, capacity=1000)
    assert total == 700 * nq and len(hits) == 1000


def test_several_parts_per_wave_slot(gpu, dev):
    """40 million rows: more than one 64-group part per resident wave.  Every
    planted row is found, at its own index."""
    import torch
    n = 40_000_003
    g = torch.Generator(device="cuda").manual_seed(3)
    db = torch.randint(-(1 << 63), (1 << 63) - 1, (n, 4), generator=g, device=dev).view(torch.uint8).reshape(n, 32)
    queries = synthetic.random_db(40, seed=9)
    q = torch.from_numpy(queries).to(dev)
    at = torch.linspace(0, n - 1, 1000, dtype=torch.float64, device=dev).round().to(torch.int64)
    db[at] = q[torch.arange(1000, device=dev) % 40]
    total, hits = gpu.match(db, q, 31, plane=gpu.build_prefix_plane(db))
    assert total == 1000
    assert np.array_equal(hits["index"].astype(np.int64), at.cpu().numpy())
    assert np.array_equal(hits["query"], np.arange(1000) % 40)


@pytest.mark.parametrize("cap", [0, 16])
def test_full_groups_over_many_rows(gpu, dev, cap):
    """1000 queries x 8 million rows run the shared-rows layout; with room for
    16 records only, its recheck matches every item again.  Both give the
    vector-ALU matcher's set."""
    import torch
    n, nq = 8_000_001, 1000
    g = torch.Generator(device="cuda").manual_seed(4)
    db = torch.randint(-(1 << 63), (1 << 63) - 1, (n, 4), generator=g, device=dev).view(torch.uint8).reshape(n, 32)
    q = torch.from_numpy(synthetic.random_db(nq, seed=10)).to(dev)
    at = torch.randperm(n, generator=g, device=dev)[:2000]
    db[at] = q[torch.arange(2000, device=dev) % nq] ^ (torch.randint(0, 256, (2000, 1), generator=g, device=dev)
                                                       .to(torch.uint8))
    gpu.set_match_record_cap(cap)
    try:
        plane = gpu.build_prefix_plane(db)
        n1, h1 = gpu.match(db, q, 31, plane=plane)
        n2, h2 = gpu.match(db, q, 31)
    finally:
        gpu.set_match_record_cap(0)
    n3, h3 = gpu.match(db, q, 31, path="valu")
    assert n1 == n2 == n3 > 0
    assert np.array_equal(triples(h1), triples(h3)) and np.array_equal(triples(h2), triples(h3))


@pytest.mark.parametrize("nq", [32, 33, 65, 129, 193, 257, 513, 1100])
def test_shards_around_their_groups(gpu, oracle, dev, nq):
    """Shards of one row, around one group, a round, a part: the hits of every
    shard carry its own base, at thresholds on both sides of the change of the
    products per accumulator."""
    import torch
    sizes = [1, 63, 64, 65, 255, 257, 1, 4095, 4097, 130]
    queries = synthetic.random_db(nq, seed=nq)
    parts = [planted(n, queries, 50 + i) for i, n in enumerate(sizes)]
    q = torch.from_numpy(queries).to(dev)
    s = gpu.Shards()
    try:
        for p in parts:
            s.add(p)
        for threshold in (27, 28, 63):
            n, want = oracle.match_all(np.concatenate(parts), queries, threshold)
            total, hits = s.match(q, threshold, capacity=1 << 18)
            assert total == n and np.array_equal(triples(hits), want), threshold
    finally:
        s.close()


@pytest.mark.parametrize("nq", [11, 12, 13, 15, 16, 17, 24, 31])
def test_fewer_than_two_tiles(gpu, oracle, dev, nq):
    """The matrix cores take 12 queries and more up to threshold 40; both sides
    of the line, single database and shards, against the oracle."""
    import torch
    assert gpu.match_uses_matrix_cores(nq, 40) == (nq >= 12) and not gpu.match_uses_matrix_cores(nq, 41)
    queries = synthetic.random_db(nq, seed=nq)
    q = torch.from_numpy(queries).to(dev)
    for n_rows in (1, 63, 257, 5000):
        db = planted(n_rows, queries, 70 + n_rows)
        d = torch.from_numpy(db).to(dev)
        plane = gpu.build_prefix_plane(d)
        s = gpu.Shards()
        try:
            s.add(db[:n_rows // 3 + 1])
            if n_rows > 1:
                s.add(db[n_rows // 3 + 1:])
            for threshold in (16, 31, 40, 41):
                n, want = oracle.match_all(db, queries, threshold)
                for total, hits in (gpu.match(d, q, threshold), gpu.match(d, q, threshold, plane=plane),
                                    s.match(q, threshold)):
                    assert total == n and np.array_equal(triples(hits), want), (n_rows, threshold)
        finally:
            s.close()


# every number of tiles from three to sixteen in one group, and two groups of an
# odd number, over more rows than the held-rows layout takes
@pytest.mark.parametrize("nq", [48, 49, 80, 97, 113, 129, 145, 161, 177, 193, 209, 225, 241, 280])
def test_every_width_over_many_rows(gpu, dev, nq):
    import torch
    n = 60_001 if nq <= 192 else 700_101
    g = torch.Generator(device=dev).manual_seed(nq)
    db = torch.randint(-(1 << 63), (1 << 63) - 1, (n, 4), generator=g, device=dev).view(torch.uint8).reshape(n, 32)
    q = torch.from_numpy(synthetic.random_db(nq, seed=13)).to(dev)
    at = torch.randperm(n, generator=g, device=dev)[:2000]
    db[at] = q[torch.arange(2000, device=dev) % nq] ^ (torch.randint(0, 256, (2000, 1), generator=g, device=dev)
                                                       .to(torch.uint8) & 19)
    db[0], db[n - 1] = q[0], q[nq - 1]
    plane = gpu.build_prefix_plane(db)
    for threshold in (27, 28):
        n0, h0 = gpu.match(db, q, threshold, path="valu")
        for p in (None, plane):
            n1, h1 = gpu.match(db, q, threshold, plane=p)
            assert n0 == n1 > 0 and np.array_equal(triples(h0), triples(h1)), (threshold, p is not None)
