"""The threshold search where coefficients lie within a few ulps of each other.

A guess is the mean of rounded sums and can fall behind the bound it replaces;
the range [mn, mx] then widens again, and the elements between are candidates
once more.  The planes here are solved (tent and DCT are linear, of rank 16) so
that most of the 256 coefficients share one value up to rounding."""
import numpy as np
import pytest

f32 = np.float32


def tree8(v):
    for _ in range(3):
        v = v[..., 0::2] + v[..., 1::2]
    return v[..., 0]


def search(p, widens=True):
    """The search as the block kernels run it -- elements leave the range for
    good, and are taken anew where a bound moves back (`widens`) -- as
    (threshold, bits' guess, whether a bound moved back)."""
    p = np.asarray(p, f32).reshape(32, 8)
    mn, mx = p.min(), p.max()
    over_in, under_in = p <= mx, p >= mn
    guess = last = f32((mn + mx) * f32(0.5))
    over = under = 0
    moved = False
    for _ in range(32):
        above, below = (p > guess) & over_in, (p < guess) & under_in
        sums = [f32(0)] * 2
        for k, m in enumerate((above, below)):
            s = np.zeros(8, f32)
            for c in range(32):
                s = s + np.where(m[c], p[c], f32(0))
            sums[k] = tree8(s)
        a, b = int(above.sum()), int(below.sum())
        last = guess
        if a + over > 128:
            under += b
            back = not guess >= mn
            mn = guess
            under_in &= ~(p < guess)
            guess = f32(sums[0] / f32(a))
        elif b + under > 128:
            over += a
            back = not guess <= mx
            mx = guess
            over_in &= ~(p > guess)
            guess = f32(sums[1] / f32(b))
        else:
            break
        moved |= back
        if back and widens:
            over_in, under_in = p <= mx, p >= mn
    return guess, last, moved


def hash_of(p, guess):
    return np.packbits(np.asarray(p, f32).reshape(32, 8) > guess, axis=1, bitorder="little")[::-1, 0]


def close_sets(n, seed):
    rng = np.random.default_rng(seed)
    for _ in range(n):
        base = f32(rng.uniform(0.5, 2))
        yield (base + np.spacing(base) * rng.integers(-12, 13, 256)).astype(f32)


def test_search_rule_over_close_coefficients(oracle):
    moved = 0
    for p in close_sets(1500, 7):
        thr, last, back = search(p)
        h, t = oracle.quantize_avx2(p)
        assert thr == f32(t) and np.array_equal(hash_of(p, last), h)
        moved += back
    assert moved >= 5  # the sets do reach the widening range


def test_widening_matters(oracle):
    """Elements that leave for good give other thresholds or bits."""
    wrong = 0
    for p in close_sets(1500, 7):
        h, t = oracle.quantize_avx2(p)
        thr, last, _ = search(p, widens=False)
        wrong += not (thr == f32(t) and np.array_equal(hash_of(p, last), h))
    assert wrong >= 3


def solved_planes(oracle, seeds):
    """One f32 plane per (free, seed): all coefficients share a value but
    `free` of them."""
    dct = oracle.tables()[1][:16 * 127].reshape(16, 127)
    tent = np.zeros((127, 512))
    for o in range(127):
        tent[o, 4 * o + 1:4 * o + 8] = np.array([0, 1, 2, 3, 2, 1, 0]) / 9.0
    inv = np.linalg.pinv(dct @ tent)
    planes = []
    for free, seed in seeds:
        rng = np.random.default_rng(seed)
        v = rng.uniform(0.5, 4)
        want = np.full(256, v)
        want[rng.permutation(256)[:free]] += rng.normal(0, v, free)
        planes.append(inv @ want.reshape(16, 16) @ inv.T)
    return np.stack(planes).astype(f32)


# planes whose NORMAL or FLOPPED search moves a bound back, and the ones around them
SEEDS = [(0, 15), (0, 133), (8, 18), (8, 80), (40, 7), (40, 55), (40, 104), (40, 113), (40, 123), (40, 149),
         (100, 11), (100, 21), (100, 31), (100, 90), (100, 129)] + [(40, s) for s in range(200, 217)]


def test_planes_reach_the_widening_range(oracle):
    moved = 0
    for x in solved_planes(oracle, SEEDS):
        moved += search(oracle.hash_get_threshold(x)[3])[2]
    assert moved >= 5


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["AUTO", "WAVE", "BLOCK4", "BLOCK8", "BLOCK16"])
def test_close_coefficients(gpu, oracle, dev, layout):
    import torch
    planes = solved_planes(oracle, SEEDS)
    h, q, t = (y.cpu().numpy() for y in gpu.hash_batch(torch.from_numpy(planes).to(dev),
                                                       layout=getattr(gpu, "LAYOUT_" + layout)))
    for k, x in enumerate(planes):
        H, Q, T, _ = oracle.hash_dihedrals(x, 1)
        assert np.array_equal(h[k], H), f"plane {SEEDS[k]}"
        assert np.array_equal(q[k], Q) and np.array_equal(t[k], T), f"plane {SEEDS[k]}"
