"""A handle's workspace: a captured step of a small domain holds the address of
the handle's first workspace, which stays where it is while larger domains make
the handle's other workspace grow and move; and the allocation-free steps of
small domains on two handles share nothing."""
import pytest

from mam4xx_amd import layout as L
from mam4xx_amd import scenes

pytestmark = pytest.mark.gpu
DT = 1800.0


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    return torch


def _scene(torch, ncol, nlev, seed):
    from mam4xx_amd.chain import scene_to_device
    d = scene_to_device(scenes.generate(ncol, nlev, seed=seed))
    return d, torch.full((L.NSTATE, nlev, ncol), float("nan"), dtype=torch.float64, device="cuda")


@pytest.mark.parametrize("ncol,nlev", [(16, 72), (256, 64)])  # 256 x 64: the most it holds
def test_captured_small_step_survives_growth(torch_cuda, ncol, nlev):
    from mam4xx_amd.chain import Chain
    torch = torch_cuda
    ch, ref = Chain(), Chain()
    d, out = _scene(torch, ncol, nlev, 31)
    _, want = _scene(torch, ncol, nlev, 31)
    ref.compute_tendencies(d, DT, want)
    ch.compute_tendencies(*_larger(torch, 301))  # the other workspace exists at the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ch.compute_tendencies(d, DT, out)
    for larger in (1200, 2400):
        ch.compute_tendencies(*_larger(torch, larger))
        for _ in range(2):
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
    del graph
    ch.close()
    ref.close()


def test_noalloc_small_steps_of_two_handles_overlap(torch_cuda):
    """each handle on a stream of its own, nothing ordering the two"""
    from mam4xx_amd.chain import Chain
    torch = torch_cuda
    ref = Chain()
    jobs = []
    for i, ncol in enumerate((96, 200)):
        d, want = _scene(torch, ncol, 72, 40 + i)
        ref.compute_tendencies(d, DT, want)
        torch.cuda.synchronize()
        jobs.append((Chain(), torch.cuda.Stream(), d, want,
                     [torch.full_like(want, float("nan")) for _ in range(8)]))
    torch.cuda.synchronize()
    for k in range(8):
        for ch, stream, d, _, outs in jobs:
            with torch.cuda.stream(stream):
                ch.compute_tendencies(d, DT, outs[k], noalloc=True)
    torch.cuda.synchronize()
    for ch, _, _, want, outs in jobs:
        for out in outs:
            assert torch.equal(out, want)
        ch.close()
    ref.close()


def _larger(torch, ncol):
    d, out = _scene(torch, ncol, 72, 32)
    return d, DT, out
