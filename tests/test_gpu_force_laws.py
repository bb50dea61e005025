"""k_forces on tissues that mix every cell state, so that the lanes of one
wave take different laws (each of cell_interaction.cpp:77-294, a DER-DER pair
twice), against the oracle's serial loop: positions equal bit for bit."""
import numpy as np
import pytest

from epi_amd.configs import ALIVE, DEAD, DER, FIX, MUSUME, AIR

from helpers import sheet_spec

pytestmark = pytest.mark.gpu


def mixed(seed, pitch, der_layers):
    """lattice layers over a dense sheet: DER cells first (index order), then
    a shuffle of the other states, two of them division partners"""
    r = np.random.default_rng(seed)
    L, side = 16.0, int(16.0 / pitch)
    free = []
    for layer in range(der_layers + 3):
        for k in range(side * side):
            state = DER if layer < der_layers else int(r.choice([ALIVE, ALIVE, DEAD, AIR, FIX, MUSUME, MUSUME]))
            j = r.uniform(-0.12, 0.12, 3)
            # DER cells from the sheet's side (z < radius meets the wall), the rest above them
            free.append(dict(state=state, x=float((k % side + 0.5) * L / side + j[0]),
                             y=float((k // side + 0.5) * L / side + j[1]), z=float(2.9 + 2.0 * layer + j[2]),
                             radius=float(r.choice([1.2, 1.4])), agek=float(r.choice([1.0, 3.5, 20.0])),
                             rest_div_times=int(r.integers(0, 3))))
    nder = der_layers * side * side
    for a in (nder, nder + 7, len(free) - 3):   # partners: lower and higher index, in and out of each other's list
        b = a + 1 if a != nder + 7 else len(free) - 5
        for p, q in ((a, b), (b, a)):
            free[p].update(state=MUSUME, pair=q, spr_nat_len=0.9)
    spec = sheet_spec(free, nmx=16, nmy=16, L=L, grid=(16, 16, 24), lz=24.0)
    spec["nder"] = nder
    spec["cells"]["z"][:spec["nmemb"]] += r.uniform(-0.05, 0.05, spec["nmemb"])
    return spec


@pytest.mark.parametrize("seed,pitch,der_layers", [(1, 2.0, 1), (2, 2.3, 2), (3, 2.0, 0)])
def test_mixed_states_match_the_serial_loop(oracle_mod, seed, pitch, der_layers):
    from epi_amd import native
    spec = mixed(seed, pitch, der_layers)
    gt, ot = native.Tissue(spec["geometry"]), oracle_mod.OracleTissue(spec["geometry"])
    for t in (gt, ot):
        t.load(spec)
    for _ in range(3):
        for t in (gt, ot):
            t.cell_interaction()
            t.pos_copy()
            t.cell_pos_periodic_fix()
            t.connect_cell()
    assert gt.error() == ot.error() == 0
    g, o = gt.get_cells(), ot.get_cells()
    assert np.array_equal(g["conn"], o["conn"])
    for k in "xyz":
        assert np.array_equal(g[k], o[k]), (k, float(np.max(np.abs(g[k] - o[k]))))
    gt.close()
