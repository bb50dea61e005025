"""cell_state_renew past its chunks, against the oracle's loop: more division-ready
cells than one round of the ordered walk takes (1,024), with divisions on both
sides of the round's end; and a tissue that outgrows the one-launch form's chunk
(1,024 cells) between two status read-backs, so that the form chosen from the
last known count walks a second chunk.  Cells, links and draws are equal."""
import numpy as np
import pytest

from epi_amd import configs

pytestmark = pytest.mark.gpu

EXACT = ("state", "pair", "dermis", "uid", "rest_div_times", "fix_origin", "conn", "x", "y", "z", "spr_nat_len", "radius")
ROUNDED = ("agek", "ageb", "in_fat", "ex_fat")   # laws with tanh: a different library's rounding


def tissue(seed, side, free, layers):
    box = 2.0 * np.ceil(0.4 * side)
    s = configs.make_tissue(seed, nmx=side, nmy=side, lx=box, ly=box, nx=int(box), ny=int(box), nz=24, n_fix=16,
                            n_free=free, n_layers=layers, lz=24.0)
    c = s["cells"]
    c["ageb"][(c["state"] == configs.MUSUME) | (c["state"] == configs.FIX)] = 40.0
    return s


def both(oracle_mod, spec, draws, params=None):
    from epi_amd import native
    o, t = oracle_mod.OracleTissue(spec["geometry"]), native.Tissue(spec["geometry"])
    for x in (o, t):
        if params:
            x.set_params(params)
        x.load(spec)
        x.set_rng(draws)
    return o, t


def equal(o, t):
    a, b = t.get_cells(), o.get_cells()
    assert o.error() == 0 and t.error() == 0
    assert a["n"] == b["n"] and t.rng_cursor() == o.rng_cursor()
    for f in EXACT:
        assert np.array_equal(a[f], b[f]), f
    for f in ROUNDED:
        assert np.allclose(a[f], b[f], rtol=1e-12, atol=1e-15), f
    return b


def test_more_ready_cells_than_a_round(oracle_mod):
    from epi_amd import native
    spec = tissue(3, 92, 2600, 2)
    r = np.random.default_rng(3)
    draws = r.uniform(0, 1, 50000)
    draws[r.uniform(0, 1, draws.size) < 0.1] *= 1e-4    # these decide for a division
    o, t = both(oracle_mod, spec, draws)
    before = o.get_cells()
    start, n = spec["nmemb"], before["n"]
    stem = np.isin(before["state"], (configs.MUSUME, configs.FIX)) & (before["dermis"] >= 0)
    ready = np.nonzero(stem)[0]
    assert ready.size > 1024 and ready[0] >= start
    do, dg = oracle_mod.Driver(0, 0, 0, 0, 0), native.Driver(0, 0, 0, 0, 0)
    o.step(do)
    t.step(dg, 1)
    after = equal(o, t)
    rank = np.searchsorted(ready, after["pair"][n:])    # the parents' places among the ready cells
    assert np.any(rank < 1024) and np.any(rank >= 1024)
    t.close()


def test_one_launch_form_past_its_chunk(oracle_mod):
    spec = tissue(4, 46, 686, 2)
    start, n0 = spec["nmemb"], spec["cells"]["x"].size
    assert n0 - start + 64 <= 768
    r = np.random.default_rng(4)
    draws = r.uniform(0, 1, 20000)
    draws[0:1200:3] *= 1e-4                             # the first renewal: every ready cell divides
    late = draws[1200:]
    late[r.uniform(0, 1, late.size) < 0.3] *= 1e-4
    # pairs part in the second renewal, and whatever has aged once is ready
    o, t = both(oracle_mod, spec, draws, dict(eps_L=1000.0, unpair_dist_coef=0.0, agki_max=0.1, stoch_div_time_ratio=0.999))
    for x in (o, t):                                    # no call here reads the count back
        x.cell_state_renew()
        x.cell_state_renew()
        x.connect_cell()
    oc = o.get_cells()
    assert oc["n"] - start > 1024
    last = np.arange(oc["n"]) >= start + 1024
    assert np.any(last & (oc["pair"] < 0) & (oc["dermis"] >= 0) & (oc["state"] == configs.MUSUME))
    for x in (o, t):
        x.cell_state_renew()
    after = equal(o, t)
    parents = after["pair"][oc["n"]:]
    assert np.any(parents >= start + 1024) and np.any(parents < start + 1024)
    t.close()
