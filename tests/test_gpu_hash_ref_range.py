"""The precise kernel on f32 planes outside the range of its fast division by
three: the passes divide instead, bit for bit as the oracle, and such planes
take no multiple of the time of others."""
import numpy as np
import pytest

from yume_pdq import synthetic

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return bool(np.all((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))))


# whole planes and single rows of each run of 64, among planes inside the range;
# the scales take the sums through the subnormals and up to overflow
@pytest.mark.parametrize("what", ["scaled down", "scaled up", "one row", "nonfinite"])
def test_planes_outside_the_range(gpu, oracle, dev, what):
    import torch
    rng = np.random.default_rng(17)
    planes = synthetic.images_u8(10, start=60).astype(np.float32) + rng.uniform(0, 1, (10, 512, 512)).astype(np.float32)
    for k in range(1, 10):
        if what == "scaled down":
            planes[k] = np.ldexp(planes[k], -20 * k).astype(np.float32)
        elif what == "scaled up":
            planes[k] = np.ldexp(planes[k] - 100, 90 + 4 * k).astype(np.float32)
        elif what == "one row":
            planes[k, 64 * (k % 8) + 7 * k, rng.integers(512)] = [1e-9, -1e-30, 2e38][k % 3]
        else:
            planes[k, 64 * (k % 8) + 7 * k, rng.integers(512)] = [np.nan, np.inf, -np.inf][k % 3]
    h, q, t, f = (y.cpu().numpy() for y in gpu.hash_ref_batch(torch.from_numpy(planes).to(dev), want_pdqf=True))
    for k in range(10):
        H, T, Q, P = oracle.hash_ref32(planes[k])
        assert same(f[k], P), k
        assert np.array_equal(h[k], H), k
        assert same(q[k], Q) and same(t[k], T), k


def test_outside_the_range_costs_no_multiple(gpu, dev):
    import torch
    planes = torch.rand((32, 512, 512), device=dev) * 255

    def once():
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            gpu.hash_ref_batch(planes)
        b.record()
        b.synchronize()
        return a.elapsed_time(b)

    inside = min(once() for _ in range(4))
    planes[:, 5, 5] = 1e-9
    outside = min(once() for _ in range(4))
    assert outside < 2.5 * inside, (outside, inside)
