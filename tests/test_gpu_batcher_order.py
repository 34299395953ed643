"""What Batcher.run(sync=False) leaves to its caller: on return the planes have
been taken and the batch before is done, whatever was still on the context's
stream at the call."""
import pytest

from yume_pdq import synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture
def context(gpu, dev):
    import torch
    s = gpu.Shards()
    s.add(torch.from_numpy(synthetic.random_db(1000, seed=5)).to(dev))
    b = gpu.Batcher(s, 64, threshold=20)
    a = torch.ones((4096, 4096), dtype=torch.float32, device=dev)
    c = torch.empty_like(a)
    torch.cuda.synchronize()

    def backlog():
        """Some milliseconds of work on the context's stream."""
        with torch.cuda.stream(b.stream):
            for _ in range(4):
                torch.mm(a, a, out=c)

    yield b, backlog
    b.close()
    s.close()


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("then", ["overwrite", "free"])
def test_planes_are_taken_on_return(gpu, dev, context, then, use_graph):
    import torch
    b, backlog = context
    base = torch.from_numpy(synthetic.images_u8(64)).to(dev)
    sizes = [1, 64, 5, 33]
    want = [gpu.hash_batch((base[:n] + 7 * k).contiguous())[0] for k, n in enumerate(sizes)]
    torch.cuda.synchronize()
    got = []
    for k, n in enumerate(sizes):
        backlog()
        planes = base[:n] + 7 * k
        b.run(planes, use_graph=use_graph, sync=False)
        if then == "overwrite":
            planes.fill_(77)
        else:
            del planes
            again = torch.empty((n, 512, 512), dtype=torch.uint8, device=dev)
            again.fill_(77)
        torch.cuda.current_stream().synchronize()
        with torch.cuda.stream(b.stream):
            got.append(b.hashes[:n].clone())
    b.stream.synchronize()
    for g, w in zip(got, want):
        assert torch.equal(g, w)


def test_previous_batch_is_done_on_return(dev, context):
    import torch
    b, backlog = context
    planes = torch.from_numpy(synthetic.images_u8(64)).to(dev)
    b.run(planes)
    for _ in range(3):
        backlog()
        b.run(planes, sync=False)
        done = torch.cuda.Event()
        done.record(b.stream)
        b.run(planes[:5], sync=False)
        assert done.query()
