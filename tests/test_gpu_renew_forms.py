"""cell_state_renew where its launch form changes (one launch or two: the counts
past the membrane on both sides of the limit) and where its chunks end, with many divisions and removals in a step, against the oracle's loop:
every cell field, the removal records and the draws consumed are equal."""
import numpy as np
import pytest

from epi_amd import configs

pytestmark = pytest.mark.gpu

# (sheet side, cells past the membrane): limit 768 - 64 of the one
# launch, chunks of 1024 and blocks of 256
SHAPES = [(16, 255), (24, 703), (24, 705), (28, 1025), (36, 2049), (44, 3007), (44, 3010), (52, 4400)]


@pytest.mark.parametrize("side,free", SHAPES)
def test_forms(oracle_mod, side, free):
    from epi_amd import native
    layers = max(3, int(np.ceil(free / (0.9 * (0.4 * side) ** 2))))
    spec = configs.config_tiny(5, n_free=free - 4, side=side, grid=side, n_layers=layers, dead_top=True,
                               nz=2 * layers + 16)
    c = spec["cells"]
    r = np.random.default_rng(free)
    dead = np.nonzero(c["state"] == configs.DEAD)[0]
    gone = np.sort(r.choice(dead[:-min(120, dead.size // 2)], min(90, dead.size // 4), replace=False))
    c["agek"][gone] = 31.4
    stem = np.nonzero((c["state"] == configs.MUSUME) | (c["state"] == configs.FIX))[0]
    c["ageb"][stem[::2]] = 40.0
    draws = r.uniform(0, 1, 200000)
    draws[r.uniform(0, 1, draws.size) < 0.1] *= 1e-4    # these decide for a division
    o, t = oracle_mod.OracleTissue(spec["geometry"]), native.Tissue(spec["geometry"])
    do, dg = oracle_mod.Driver(7, 0, 0, 0, 0), native.Driver(7, 0, 0, 0, 0)
    for x in (o, t):
        x.load(spec)
        x.set_rng(draws)
    n0 = c["x"].size
    print(f"renewal forms: {free} cells past the membrane", flush=True)
    for k in range(3):
        o.step(do)
        t.step(dg, 1)
        assert o.error() == 0 and t.error() == 0, k
        a, b = t.get_cells(), o.get_cells()
        assert a["n"] == b["n"] and t.rng_cursor() == o.rng_cursor(), k
        for f in ("state", "pair", "dermis", "uid", "rest_div_times", "fix_origin", "conn", "x", "y", "z",
                  "spr_nat_len", "radius"):
            assert np.array_equal(a[f], b[f]), (k, f)
        for f in ("agek", "ageb", "in_fat", "ex_fat"):   # laws with tanh: a different library's rounding
            assert np.allclose(a[f], b[f], rtol=1e-12, atol=1e-15), (k, f)
    assert o.get_cells()["uid"].max() >= n0   # divisions happened
    g, w = t.take_cell_stats(), o.take_cell_stats()
    assert np.array_equal(g, w) and len(g) > 0
    t.close()
