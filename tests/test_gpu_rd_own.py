"""The reverse sub-step where a cell owns few voxels, more than one sweep of
its lanes takes, and none (DEAD cells and cells above the box), against the
oracle's reverse pass.  Tolerances as for the other gradients: FP64 sums in
another order, 1e-8."""
import numpy as np
import pytest

from epi_amd import configs

pytestmark = pytest.mark.gpu

# (grid points per edge of a 16-wide box, planes, dead top layer)
SHAPES = [(13, 20, False), (20, 28, True), (40, 56, False), (48, 64, True)]


@pytest.mark.parametrize("grid,nz,dead", SHAPES)
def test_owned_voxels(oracle_mod, grid, nz, dead):
    from epi_amd import native
    spec = configs.config_tiny(11, n_free=240, side=20, grid=grid, n_layers=3 if dead else 2, dead_top=dead, nz=nz)
    g = spec["geometry"]
    o = oracle_mod.OracleTissue(g)
    o.load(spec)
    t = native.Tissue(g)
    t.load(spec)
    zz = t.calc_zzmax()
    n = t.get_cells()["state"].size
    n_sub = 6
    base = dict(du=0.0104, dp=0.096, gj0=0.97, kpa=np.full(n, 5.0))
    tgt = o.rd_forward(zz, n_sub, du=0.011, dp=0.09, gj0=0.93, kpa=np.full(n, 5.3))
    lo, go = o.rd_adjoint(zz, n_sub, tgt, **base)
    t.set.rd_begin(zz)
    for lanes in (8, 16):
        print(f"rd adjoint: {grid}x{grid}x{nz}, dead {dead}, {lanes} lanes per cell", flush=True)
        t.set.set_tuning({"rd_group": lanes})
        loss, grads = t.set.rd_adjoint([base], n_sub, 4, [tgt])
        assert loss[0] == pytest.approx(lo, rel=1e-10)
        for k in ("du", "dp", "gj0"):
            assert grads[0][k] == pytest.approx(go[k], rel=1e-8), k
        sel = np.abs(go["kpa"]) > 1e-3 * np.max(np.abs(go["kpa"]))
        assert np.max(np.abs(grads[0]["kpa"][sel] - go["kpa"][sel]) / np.abs(go["kpa"][sel])) <= 1e-8
    t.set.rd_end()
