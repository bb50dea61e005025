"""setup_map_lat on stamp boxes of every shape the lanes' walk has: narrower
and wider than the lane count, cut by the grid's floor and top, across the
periodic planes and their copies, each with every lane count, against the
oracle's serial stamping (map.cpp:18-167); maps and lattice points equal."""
import numpy as np
import pytest

from epi_amd.configs import ALIVE, DEAD, FIX, MUSUME

from helpers import sheet_spec

pytestmark = pytest.mark.gpu

L, LZ = 14.0, 18.0


def spec_on(grid, seed):
    r = np.random.default_rng(seed)
    free = [dict(state=int(r.choice([ALIVE, DEAD, FIX, MUSUME])), x=float(r.uniform(0, L)), y=float(r.uniform(0, L)),
                 z=float(z), radius=float(r.choice([0.9, 1.4])))
            for z in np.concatenate([r.uniform(2.5, LZ - 3, 60), [0.2, LZ - 0.3, LZ - 1.0]])]
    # corners and seams of the box
    for x, y in ((0.0, 0.0), (np.nextafter(L, 0), np.nextafter(L, 0)), (0.0, 7.0), (7.0, 0.01), (L - 0.01, 3.0)):
        free.append(dict(state=ALIVE, x=float(x), y=float(y), z=6.0))
    return sheet_spec(free, L=L, grid=grid, lz=LZ)


@pytest.mark.parametrize("lanes", [1, 4, 16])
@pytest.mark.parametrize("grid", [(14, 14, 18), (33, 21, 25), (9, 11, 12), (60, 57, 70), (6, 6, 8)])
def test_stamps_match_the_oracle(oracle_mod, grid, lanes):
    from epi_amd import native
    spec = spec_on(grid, sum(grid))
    gt, ot = native.Tissue(spec["geometry"]), oracle_mod.OracleTissue(spec["geometry"])
    gt.set.set_tuning({"map_lanes": lanes})
    for t in (gt, ot):
        t.load(spec)
        t.setup_map_lat()
        t.setup_map_lat()   # the second build clears what the first stamped
    g, o = gt.get_fields(), ot.get_fields()
    for k in ("cmap1", "cmap2"):
        assert np.array_equal(g[k], o[k]), (k, int(np.count_nonzero(g[k] != o[k])))
    assert np.array_equal(gt.get_cells()["lat"], ot.get_cells()["lat"])
    gt.close()
