"""A reaction-diffusion gradient where a tissue's capacity for cells is far larger
than its grid: the segment states are sized by what is stored of them (the grid
by the cells' averages), so that the gradient is that of the same tissue in a
context of ordinary capacity."""
import numpy as np
import pytest

from epi_amd import configs

pytestmark = pytest.mark.gpu


def gradient(cap, n_sub, every):
    from epi_amd import native
    spec = configs.config_tiny(8, n_free=220, side=20, grid=20, nz=28)
    if cap:
        spec["geometry"].max_cells = cap
    t = native.Tissue(spec["geometry"])
    t.load(spec)
    t.setup_map_lat()
    zz = t.calc_zzmax()
    t.set.rd_begin(zz)
    t.set.rd_forward([dict(du=0.0105, dp=0.095, gj0=0.94)], n_sub)
    target = t.set.rd_get_ca2p(0)
    loss, g = t.set.rd_adjoint([dict(du=0.01, dp=0.1, gj0=0.99)], n_sub, every, [target])
    t.set.rd_end()
    t.close()
    return loss[0], g[0]


@pytest.mark.parametrize("n_sub,every", [(5, 5), (6, 2)])
def test_capacity_past_the_grid(n_sub, every):
    loss, g = gradient(0, n_sub, every)
    loss2, g2 = gradient(100_000, n_sub, every)   # box: some 8,000 points
    assert loss > 0 and loss2 == pytest.approx(loss, rel=1e-12)
    for k in ("du", "dp", "gj0"):                  # FP64 atomics in another order
        assert g2[k] == pytest.approx(g[k], rel=1e-9), k
    assert np.allclose(g2["kpa"], g["kpa"], rtol=1e-9, atol=1e-9 * np.max(np.abs(g["kpa"])))
