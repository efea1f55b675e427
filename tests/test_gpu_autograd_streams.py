"""autograd.tendencies on several streams and in a captured graph."""
import pytest

from mam4xx_amd import scenes

pytestmark = pytest.mark.gpu
DT = 1800.0


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    return torch


def _job(torch, ncol, seed):
    from mam4xx_amd.chain import scene_to_device
    d = scene_to_device(scenes.generate(ncol, 72, seed=seed))
    x = [d[k].clone().requires_grad_(True) for k in ("state", "temperature", "pressure", "qv")]
    g = torch.ones_like(d["state"])
    return d, x, g


def _run(torch, job):
    from mam4xx_amd.autograd import tendencies
    d, x, g = job
    y = tendencies(*x, d, DT)
    return [y.detach()] + list(torch.autograd.grad(y, x, grad_outputs=g))


def test_streams_that_nothing_orders(torch_cuda):
    torch = torch_cuda
    jobs = [_job(torch, ncol, 50 + i) for i, ncol in enumerate((64, 300, 150))]
    want = [_run(torch, j) for j in jobs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in jobs]
    got = []
    for _ in range(3):
        for s, j in zip(streams, jobs):
            with torch.cuda.stream(s):
                got.append(_run(torch, j))
    torch.cuda.synchronize()
    for i, outs in enumerate(got):
        for a, b in zip(outs, want[i % 3]):
            assert torch.equal(a, b)


@pytest.mark.parametrize("ncol", [16, 300])  # below and above 16,384 cells
def test_warm_up_on_one_stream_and_capture_on_another(torch_cuda, ncol):
    from mam4xx_amd.autograd import tendencies
    torch = torch_cuda
    d, x, _ = _job(torch, ncol, 60)
    x = [t.detach() for t in x]
    want = tendencies(*x, d, DT)
    other = _job(torch, 200, 61)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = tendencies(*x, d, DT)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        _run(torch, other)  # the program's own work between the replays
        torch.cuda.synchronize()
