"""NaN / Inf at the places where the streamed test of f32 planes changes hands
-- the first and last rows and columns the reference reads, and the rows where
one wave's band ends and the next begins -- in every layout, and the precise
kernel's passes: planes inside and outside the range of its fast division,
mixed in one batch, against the oracle bit for bit."""
import numpy as np
import pytest

from yume_pdq import synthetic

pytestmark = pytest.mark.gpu

# bands of 8, 16 and 32 compressed rows start at input rows 32 b + 1, 64 b + 1, 128 b + 1
PLACES = [(r, c) for r in (1, 2, 3, 32, 33, 34, 64, 65, 66, 128, 129, 130, 509, 510, 511) for c in (1, 2, 511)] + \
         [(2, 0), (33, 0), (510, 0), (511, 0), (1, 256), (511, 256)]


def same(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return bool(np.all((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_nonfinite_at_edges(gpu, oracle, dev, value):
    import torch
    base = synthetic.images_u8(1, start=70)[0].astype(np.float32)
    planes = np.repeat(base[None], len(PLACES), 0)
    for k, (r, c) in enumerate(PLACES):
        planes[k, r, c] = value
    x = torch.from_numpy(planes).to(dev)
    want = [oracle.hash_dihedrals(p, 1) for p in planes]
    for layout in (gpu.LAYOUT_WAVE, gpu.LAYOUT_BLOCK4, gpu.LAYOUT_BLOCK8, gpu.LAYOUT_BLOCK16):
        h, q, t = (y.cpu().numpy() for y in gpu.hash_batch(x, layout=layout))
        for k, (H, Q, T, _) in enumerate(want):
            where = f"layout {layout}, {value} at {PLACES[k]}"
            assert np.array_equal(h[k], H), where
            assert same(q[k], Q) and same(t[k], T), where


def ref_planes(n, seed):
    """Ordinary planes, with every third one outside the fast division's
    range: a value below 2^-25, above 2^100, NaN or Inf, at a corner."""
    rng = np.random.default_rng(seed)
    planes = synthetic.images_u8(n, start=seed).astype(np.float32)
    planes += rng.uniform(0, 1, planes.shape).astype(np.float32)
    planes[0, :40, :40] = 0.0
    planes[0, 40, :] = np.float32(2.0 ** -25)  # the smallest value inside the range
    odd = [2.0 ** -26, 1e-40, 2.0 ** 101, np.nan, -np.inf]
    for k in range(1, n, 3):
        r, c = [(0, 0), (511, 511), (0, 511), (511, 0), (255, 300)][k % 5]
        planes[k, r, c] = odd[(k // 3) % 5]
    return planes


# image counts around the eight images that share a round of blocks
@pytest.mark.parametrize("n", [1, 7, 8, 9, 17])
def test_ref_passes(gpu, oracle, dev, n):
    import torch
    planes = ref_planes(n, 80 + n)
    for kind in ("f32", "u8"):
        p = planes if kind == "f32" else np.clip(np.nan_to_num(planes), 0, 255).astype(np.uint8)
        h, q, t, f = (y.cpu().numpy() for y in gpu.hash_ref_batch(torch.from_numpy(p).to(dev), want_pdqf=True))
        for k in range(n):
            H, T, Q, P = oracle.hash_ref32(p[k].astype(np.float32))
            where = f"{kind} image {k} of {n}"
            assert same(f[k], P), where
            assert np.array_equal(h[k], H), where
            assert same(q[k], Q) and same(t[k], T), where


# the scales take the threshold search's sums from subnormal over the range of
# its short division to infinity; 127 and 120 overflow in the DCT
@pytest.mark.parametrize("exponent", [None, -165, -150, -140, -120, -100, -95, -60, 0, 60, 85, 95, 110, 120, 127])
def test_threshold_search_at_all_scales(gpu, oracle, dev, exponent):
    import torch
    planes = synthetic.images_u8(3, start=90).astype(np.float32)
    planes -= np.float32(128)
    planes[2] = np.abs(planes[2])
    planes *= np.float32(2.0 ** -7)
    planes = np.zeros_like(planes) if exponent is None else np.ldexp(planes, exponent).astype(np.float32)
    if exponent is not None and exponent < -126:
        planes = np.abs(planes)  # a zero's sign may differ with negative subnormals
    x = torch.from_numpy(planes).to(dev)
    want = [oracle.hash_dihedrals(p, 1) for p in planes]
    for layout in (gpu.LAYOUT_BLOCK4, gpu.LAYOUT_BLOCK8, gpu.LAYOUT_BLOCK16):
        h, q, t = (y.cpu().numpy() for y in gpu.hash_batch(x, layout=layout))
        for k, (H, Q, T, _) in enumerate(want):
            where = f"layout {layout}, 2^{exponent}, image {k}"
            assert np.array_equal(h[k], H), where
            assert same(q[k], Q) and same(t[k], T), where


@pytest.mark.parametrize("per_cu", [1, 5.5])
def test_automatic_layout_around_its_lines(gpu, dev, per_cu):
    """Batches on both sides of a change of layout equal the wave form's."""
    import torch
    n = int(per_cu * torch.cuda.get_device_properties(dev).multi_processor_count) + 1
    x = torch.from_numpy(synthetic.images_u8(64)).to(dev).repeat((n + 63) // 64, 1, 1)[:n].contiguous()
    x[-1] = 255 - x[-1]
    want = gpu.hash_batch(x, layout=gpu.LAYOUT_WAVE)
    for m in (n, n - 1):
        got = gpu.hash_batch(x[n - m:])
        for a, b in zip(got, want):
            assert torch.equal(a, b[n - m:])


@pytest.mark.parametrize("kind", ["u8", "f32", "rgb8", "rgba8"])
def test_automatic_layout_of_small_batches(gpu, dev, kind):
    """Batches on both sides of the change from sixteen waves to eight equal the
    wave form's."""
    import torch
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    n = {"u8": cus // 32, "f32": 1, "rgb8": cus // 8 * 3, "rgba8": cus // 8}[kind] + 1
    x = torch.from_numpy(synthetic.images_u8(16)).to(dev).repeat((n + 15) // 16, 1, 1)[:n].contiguous()
    if kind == "f32":
        x = x.to(torch.float32) * 0.75
    elif kind != "u8":
        x = torch.stack([x, 255 - x, x // 2, x][:3 if kind == "rgb8" else 4], 3).contiguous()
    want = gpu.hash_batch(x, layout=gpu.LAYOUT_WAVE)
    for m in (n, n - 1):
        for a, b in zip(gpu.hash_batch(x[n - m:]), want):
            assert torch.equal(a, b[n - m:])
