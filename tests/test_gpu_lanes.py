"""No lane of a wave shows in another's results.  Cells of all three cloud
categories (clear, partly cloudy, overcast) side by side in every wave against
the same cells one call each, where a wave has one lane and every branch is
uniform: bit for bit, for every kernel of the chain that keeps values in
accumulation registers (build.py, ACC_KERNELS) and every output it writes.  A
compiler that moves such a value inside a divergent branch, and leaves out the
lanes that are off there, shows here."""
import numpy as np
import pytest

from mam4xx_amd import _abi
from mam4xx_amd import layout as L
from mam4xx_amd import scenes

pytestmark = pytest.mark.gpu
DT = 1800.0
NLEV, NCOL = 3, 43  # 129 cells: two waves and a lane
PLANES = ("state", "temperature", "pressure", "height", "qv", "cloud_fraction", "dgncur_a",
          "dgncur_awet", "wetdens")


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    return torch


@pytest.fixture(scope="module")
def cells(torch_cuda):
    """the scene and a second state (before the cloud chemistry) on the GPU, and
    a direction"""
    from mam4xx_amd.chain import scene_to_device
    sc = scenes.generate(NCOL, 72, seed=81)
    r = np.random.default_rng(82)
    lev = [20, 45, 70]
    sc = {k: (np.ascontiguousarray(v[..., lev, :]) if v.ndim > 1 else v) for k, v in sc.items()}
    cat = r.integers(0, 3, (NLEV, NCOL))
    sc["cloud_fraction"] = np.choose(cat, [0.0, r.uniform(0.05, 0.95, cat.shape), 0.9995])
    for row in cat.reshape(-1)[:128].reshape(2, 64):
        assert len(set(row)) == 3
    d = scene_to_device(sc)
    gpu = lambda a: torch_cuda.as_tensor(np.ascontiguousarray(a)).cuda()  # noqa: E731
    x = d["state"].shape
    return (d, gpu(sc["state"] * r.uniform(0.5, 1.0, x)), gpu(sc["state"] * r.standard_normal(x)),
            gpu(r.standard_normal(x)))


def _take(t, k, j):
    """cell (k, j) of [..., level, column], or of [column]"""
    return (t[..., k:k + 1, j:j + 1] if t.dim() > 1 else t[j:j + 1]).contiguous()


def _outputs(torch, run, ch, cells, pre, cell=None):
    """a run's outputs on all cells, or on one"""
    d, p, v, g = cells
    if cell:
        d = {k: _take(t, *cell) if k in PLANES + ("pblh",) else t for k, t in d.items()}
        p, v, g = (_take(t, *cell) for t in (p, v, g))
    return run(torch, ch, d, p if pre else None, v, g)


def _new(torch, d, *lead):
    return torch.full(lead + tuple(d["temperature"].shape), float("nan"), dtype=torch.float64,
                      device="cuda")


def step(diag=False, batch=False, **cfg):
    def run(torch, ch, d, pre, v, g):
        new = lambda: [_new(torch, d, n) for n in (L.NSTATE, L.NSTATE, 4, 4)]  # noqa: E731
        o = new()
        if batch:
            both = list(zip(o, new()))
            b = ch.batch([d, d], DT, both[0], state_out=both[1], dgn_i=both[2], dgn_c=both[3])
            b.run()
            torch.cuda.synchronize()
            b.close()
            return o
        cap = torch.full(d["temperature"].shape, -1, dtype=torch.int32, device="cuda")
        proc = _new(torch, d, 5, 31) if diag else None
        ch.compute_tendencies(d, DT, o[0], state_out=o[1], dgn_i=o[2], dgn_c=o[3],
                              precldchem=pre, soa_capped=cap, process=proc)
        return o + [cap] + ([proc] if diag else [])
    return run, cfg


def tangent(**cfg):
    def run(torch, ch, d, pre, v, g):
        o = [_new(torch, d, L.NSTATE), _new(torch, d, L.NSTATE)]
        ch.compute_tangent(d, DT, o[0], o[1], dstate=v, dtemperature=d["temperature"] * 1e-3,
                           dqv=d["qv"] * 1e-2, precldchem=pre)
        return o
    return run, cfg


def adjoint(**cfg):
    def run(torch, ch, d, pre, v, g):
        o = [_new(torch, d, L.NSTATE)] + [_new(torch, d) for _ in range(3)]
        ch.compute_adjoint(d, DT, g, state_bar=o[0], temperature_bar=o[1], pressure_bar=o[2],
                           qv_bar=o[3], precldchem=pre)
        return o
    return run, cfg


FUSED, QUEUE, MIXED = _abi.SCHED_FUSED, _abi.SCHED_QUEUE, _abi.PREC_MIXED
# runs whose common outputs are the same step's, bit for bit
SAME = {
    "step": [step(schedule=QUEUE), step(schedule=FUSED), step(True, schedule=QUEUE),
             step(True, schedule=FUSED), tangent()],
    "sub-steps": [step(schedule=QUEUE, ntsubstep=3), step(schedule=FUSED, ntsubstep=3),
                  step(True, schedule=QUEUE, ntsubstep=3),
                  step(True, schedule=FUSED, ntsubstep=3), tangent(ntsubstep=3)],
    "mixed": [step(schedule=QUEUE, precision=MIXED), step(schedule=FUSED, precision=MIXED)],
    "mixed sub-steps": [step(schedule=QUEUE, precision=MIXED, ntsubstep=3),
                        step(schedule=FUSED, precision=MIXED, ntsubstep=3)],
    "no condensation": [step(schedule=QUEUE, do_cond=0), step(True, do_cond=0),
                        tangent(do_cond=0)],
    "no condensation, sub-steps": [step(do_cond=0, ntsubstep=3), tangent(do_cond=0, ntsubstep=3)],
    "adjoint": [adjoint()],
    "adjoint, sub-steps": [adjoint(ntsubstep=3)],
    "adjoint, no condensation": [adjoint(do_cond=0)],
}
BATCH = {
    "step": [step(schedule=QUEUE), step(batch=True, schedule=QUEUE),
             step(batch=True, schedule=FUSED)],
    "sub-steps": [step(schedule=QUEUE, ntsubstep=3), step(batch=True, ntsubstep=3)],
    "mixed": [step(schedule=QUEUE, precision=MIXED), step(batch=True, precision=MIXED),
              step(batch=True, schedule=FUSED, precision=MIXED)],
    "mixed sub-steps": [step(schedule=QUEUE, precision=MIXED, ntsubstep=3),
                        step(batch=True, precision=MIXED, ntsubstep=3)],
}


def _check(torch, runs, cells, pre):
    from mam4xx_amd.chain import Chain
    first = None
    for i, (run, cfg) in enumerate(runs):
        ch = Chain(**cfg)
        whole = [t.cpu() for t in _outputs(torch, run, ch, cells, pre)]
        assert all(bool(torch.isfinite(t).all()) for t in whole)
        first = first or whole
        for a, b in zip(first, whole[:1] if len(whole) == 2 else whole):  # a tangent: the values
            assert torch.equal(a, b), ("another step's results", i)
        for k in range(NLEV):
            for j in range(NCOL):
                one = _outputs(torch, run, ch, cells, pre, (k, j))
                for n, (t, u) in enumerate(zip(whole, one)):
                    assert torch.equal(t[..., k, j], u[..., 0, 0].cpu()), (i, n, k, j)
        ch.close()


@pytest.mark.parametrize("pre", [False, True], ids=["", "before cloud chemistry"])
@pytest.mark.parametrize("what", list(SAME))
def test_cells_do_not_see_their_neighbours(torch_cuda, cells, what, pre):
    _check(torch_cuda, SAME[what], cells, pre)


@pytest.mark.parametrize("what", list(BATCH))
def test_batched_cells_do_not_see_their_neighbours(torch_cuda, cells, what):
    _check(torch_cuda, BATCH[what], cells, False)
