"""connect_cell where buckets hold few and many cells: around the seven cells
of a bucket's head, past them by a whole and a part of a 16-byte load, and
with more candidates or partners than a cell's lists in the sweep hold;
neighbour rows, counts and gap junctions equal the serial build's entry for
entry, with both numbers of lanes per cell, over two builds (the second meets
buckets that the first has filled and emptied, and cells that have moved)."""
import numpy as np
import pytest

from epi_amd.configs import ALIVE, DEAD

from helpers import sheet_spec

pytestmark = pytest.mark.gpu


def crowd(seed, per_cluster, scatter, radius):
    r = np.random.default_rng(seed)
    L = 16.0
    at = []
    # clusters well inside one bucket, in a shuffled index order
    for k, m in enumerate(per_cluster):
        centre = np.array([3.0 + 4.0 * (k % 4), 3.0 + 4.0 * (k // 4 % 4), 5.0])
        at += [centre + r.uniform(-0.35, 0.35, 3) for _ in range(m)]
    at += [np.array([r.uniform(0, L), r.uniform(0, L), r.uniform(3.0, 12.0)]) for _ in range(scatter)]
    order = r.permutation(len(at))
    free = [dict(state=ALIVE if i % 3 else DEAD, x=float(at[i][0]), y=float(at[i][1]), z=float(at[i][2]),
                 radius=radius, agek=1.0) for i in order]
    return sheet_spec(free, nmx=16, nmy=16, L=L, grid=(16, 16, 24), lz=24.0)


# (cells of each cluster, scattered cells, radius)
CASES = [([1, 2, 3, 4, 6, 7, 8, 9], 0, 0.8), ([10, 11, 12, 15, 16], 20, 0.6), ([64, 65, 66], 0, 0.6),
         ([120], 40, 0.5), ([20] * 16, 700, 0.45)]


@pytest.mark.parametrize("lanes", [32, 64])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_rows(oracle_mod, case, lanes):
    from epi_amd import native
    spec = crowd(case, *CASES[case])
    g = spec["geometry"]
    n = len(spec["cells"]["x"])
    # few cells take a wave each: 32 lanes need a set of many copies
    copies = 1 if lanes == 64 else 8192 // (n - spec["nmemb"]) + 1
    ts = native.TissueSet([g] * copies)
    print(f"crowded buckets {CASES[case]}, {copies} copies", flush=True)
    shift = np.where(np.arange(n) < spec["nmemb"], 0.0, np.random.default_rng(99).uniform(-0.2, 0.2, n))
    for k in range(2):
        cells = dict(spec["cells"])
        for f in "xy":
            cells[f] = (np.asarray(cells[f]) + k * shift) % 16.0
        moved = dict(spec, cells=cells)
        ot = oracle_mod.OracleTissue(g)
        ot.load(moved)
        ot.connect_cell()
        assert ot.error() == 0
        b = ot.get_cells()
        for t in range(copies):
            ts.load(t, moved)
        ts.connect_cell()
        for t in sorted({0, copies // 2, copies - 1}):
            a = ts.get_cells(t)
            for f in ("conn_ptr", "conn", "gj", "dermis"):
                assert np.array_equal(a[f], b[f]), (k, t, f)
    ts.close()
