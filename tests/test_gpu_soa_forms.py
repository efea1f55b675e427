"""The work queue's two forms of the SOA loop on the GPU -- four lanes to a cell
(small launches, and the end of every launch) and one lane to a cell -- against
the fused kernel, bit for bit, at cell counts around the forms' own sizes: 16
cells to a wave, 32 to a staged segment, 64 and 256 to a claim, the smallest
domains, and one large enough to start with a lane to a cell.  Some columns
hold SOA masses outside the range of the loop's fast quotients."""
import numpy as np
import pytest

from mam4xx_amd import layout as L
from mam4xx_amd import scenes

pytestmark = pytest.mark.gpu
DT = 1800.0


@pytest.mark.parametrize("ncol,nlev,cfg", [
    (1, 1, {}), (1, 15, {}), (1, 17, {}), (3, 11, {}), (13, 5, {}), (257, 1, {}), (16, 72, {}),
    (301, 72, {}), (301, 72, dict(soa_blocks_per_cu=1, soa_chunk=7)), (2311, 72, {}),
    (2311, 72, dict(soa_chunk=1 << 20)),
    (2311, 72, dict(soa_chunk=33, soa_short_chunk=5, soa_short_bucket=24)),
    (2311, 72, dict(soa_short_bucket=1)),
])
def test_queue_forms_equal_the_fused_kernel(ncol, nlev, cfg):
    import torch
    from mam4xx_amd import _abi
    from mam4xx_amd.chain import Chain, scene_to_device
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    sc = scenes.generate(ncol, nlev, seed=3)
    r = np.random.default_rng(4)
    soa = [L.F_SOAG] + [L.f_qi(m, s) for m in range(4) for s, sp in enumerate(L.MODE_SPECIES[m])
                        if L.SPECIES_NAMES[sp] == "soa"]
    for f in soa:  # a tenth of the columns each: tiny masses, none
        sc["state"][f][:, r.random(ncol) < 0.1] *= 1e-290
        sc["state"][f][:, r.random(ncol) < 0.1] = 0.0
    d = scene_to_device(sc)
    out = []
    for kw in (dict(schedule=_abi.SCHED_FUSED), dict(schedule=_abi.SCHED_QUEUE, **cfg), cfg):
        ch = Chain(**kw)
        t = torch.full((L.NSTATE, nlev, ncol), float("nan"), dtype=torch.float64, device="cuda")
        cap = torch.full((nlev, ncol), -1, dtype=torch.int32, device="cuda")
        for _ in range(2):  # the second step reuses the first one's workspace
            ch.compute_tendencies(d, DT, t, soa_capped=cap)
        torch.cuda.synchronize()
        out.append((t.cpu().numpy(), cap.cpu().numpy()))
        ch.close()
    for t, cap in out[1:]:
        assert np.array_equal(t.view(np.int64), out[0][0].view(np.int64))
        assert np.array_equal(cap, out[0][1])


@pytest.mark.parametrize("ncol,dt", [(3, 59.9), (3, 60.0), (227, 1.0), (227, 30.0), (228, 30.0),
                                     (911, 19.9), (911, 20.0), (1000, 0.5)])
def test_short_steps_take_the_same_values(ncol, dt):
    """either side of the rules on the step's length (72 levels: 227 columns are
    the last of fewer than 16,384 cells, 911 the first of more than 65,536)"""
    import torch
    from mam4xx_amd import _abi
    from mam4xx_amd.chain import Chain, scene_to_device
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    d = scene_to_device(scenes.generate(ncol, 72, seed=9))
    out = []
    for kw in (dict(schedule=_abi.SCHED_FUSED), dict(schedule=_abi.SCHED_QUEUE), {}):
        ch = Chain(**kw)
        t = [torch.full((L.NSTATE, 72, ncol), float("nan"), dtype=torch.float64, device="cuda")
             for _ in range(2)]
        ch.compute_tendencies(d, dt, t[0])
        b = ch.batch([d], dt, [t[1]])
        b.run()
        torch.cuda.synchronize()
        out += [x.cpu().numpy().view(np.int64) for x in t]
        b.close()
        ch.close()
    for t in out[1:]:
        assert np.array_equal(t, out[0])
