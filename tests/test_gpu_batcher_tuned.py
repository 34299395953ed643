"""A tuned context takes no longer than an untuned one where tuning chose the
matrix cores: the query groups of every batch size are as even as untuned."""
import pytest

from yume_pdq import synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("choices", ["8=valu 32=mfma:2 64=mfma:4 128=mfma:8 256=mfma:16",
                                     "8=valu 32=mfma:2 256=mfma:16"])
def test_tuned_batches_keep_the_plan(gpu, dev, tmp_path, choices):
    import torch
    g = torch.Generator(device=dev).manual_seed(5)
    rows = torch.randint(-(1 << 63), (1 << 63) - 1, (20_000_000, 4), generator=g, device=dev).view(torch.uint8)
    s = gpu.Shards()
    s.add(rows.reshape(-1, 32))
    gpu.tune_clear()
    b = gpu.Batcher(s, 64, threshold=31)
    planes = torch.from_numpy(synthetic.images_u8(64)).to(dev)

    def best(n):
        times = []
        for _ in range(12):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            b.run(planes[:n])
            start.record(b.stream)
            b.run(planes[:n], sync=False)
            end.record(b.stream)
            end.synchronize()
            times.append(start.elapsed_time(end))
        return sorted(times)[1]

    sizes = (5, 7, 12, 20, 25, 37, 50)
    try:
        untuned = {n: best(n) for n in sizes}
        results = {n: b.run(planes[:n]) for n in sizes}
        b.autotune(iterations=1)
        path = tmp_path / "tune.txt"
        gpu.tune_save(str(path))
        line = [x for x in path.read_text().splitlines() if not x.startswith("#")][0]
        path.write_text(line.split(" :")[0] + " : " + choices + "\n")
        gpu.tune_clear()
        assert gpu.tune_load(str(path)) == 1
        tuned = {n: best(n) for n in sizes}
        for n in sizes:
            got = b.run(planes[:n])
            assert got[3] == results[n][3] and (got[4] == results[n][4]).all()
        # the last bucket's choices may be as untuned or equal; none is worse
        assert all(tuned[n] < 1.12 * untuned[n] for n in sizes), (tuned, untuned)
    finally:
        b.close()
        s.close()
        gpu.tune_clear()
