"""Where it pays, the photolysis level pass puts a block's cells in an order of its
own, which must not show: a domain, its columns taken a few at a time (as they
come) and the level-fastest layout (blocked by tiles of levels and columns) give
the same bits, with domains off the block's sizes, dark columns, one cell, and
tables with more places than the order has groups."""
import numpy as np
import pytest

from mam4xx_amd import photo_tables as PT

pytestmark = pytest.mark.gpu


def rates(torch, t, cols, sel, col_lev):
    from mam4xx_amd import _abi
    from mam4xx_amd.chain import Chain
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64)).cuda()  # noqa: E731
    lay = lambda a: dev(a[:, sel].T if col_lev else a[:, sel])  # noqa: E731
    table = {k: dev(v) for k, v in t.items()}
    table["lng_index"] = 0
    photo = lay(cols["photo"])
    ch = Chain()
    ch.compute_photolysis(table, dict(pressure=lay(cols["pmid"]), pdel=lay(cols["pdel"]),
                                      temperature=lay(cols["temp"]), o3_column=lay(cols["colo3"]),
                                      liquid_water=lay(cols["lwc"]),
                                      cloud_fraction=lay(cols["clouds"])),
                          dev(cols["zen_angle"][sel]), dev(cols["srf_alb"][sel]), photo,
                          layout=_abi.LAYOUT_COL_LEV if col_lev else _abi.LAYOUT_LEV_COL)
    torch.cuda.synchronize()
    ch.close()
    r = photo.cpu().numpy()
    return r.T if col_lev else r


# the last five in order: either layout (16 MB, 120 x 547 cells), level-fastest
# (10 MB from 1,024 cells; 400 places from 65,536; a small table from 262,144)
@pytest.mark.parametrize("ncol,nlev,axes,nw", [
    (1537, 72, "wide", 5), (513, 5, "wide", 5), (700, 31, "ref", 5), (1, 1, "wide", 5),
    (129, 73, "fine", 5),
    (547, 120, "wide", 67), (129, 73, "wide", 40), (43, 24, "wide", 40), (911, 72, "fine", 4),
    (3651, 72, "ref", 5)])
def test_the_blocks_order_does_not_show(ncol, nlev, axes, nw):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    rng = np.random.default_rng(ncol)
    ax = dict(wide=PT.wide_axes(), ref=PT.REF_AXES,
              # more places than groups
              fine=PT.wide_axes(numsza=20, numcolo3=20, numalb=12))[axes]
    t = PT.random_table(rng, ax, nw=nw)
    cols = PT.columns(rng, nlev, ncol, PT.wide_axes())
    cols["temp"][:, :: 7] = rng.uniform(120.0, 380.0, cols["temp"][:, :: 7].shape)
    a = rates(torch, t, cols, np.arange(ncol), False)
    b = rates(torch, t, cols, np.arange(ncol), True)
    assert np.array_equal(a, b)
    assert (a != cols["photo"]).any() or ncol == 1
    for s in (np.arange(min(3, ncol)), np.arange(max(0, ncol - 4), ncol)):
        assert np.array_equal(a[:, s], rates(torch, t, cols, s, False))
