"""A solve of several uneven tissues that is fused and whose launches are large
enough for XCD-contiguous runs (2,048 workgroups; the list's cell blocks are
padded to a multiple of 8): as the same solve with XCD 0, as every tissue alone,
and as two launches a sub-step, bit for bit."""
import numpy as np
import pytest

from epi_amd import configs

pytestmark = pytest.mark.gpu

KEYS = ("ca2p", "ca2p_next", "ip3", "ip3_next", "ca2p_avg", "ex_inert", "gj")


def tissues():
    """three uneven tissues with odd grids, some 20,000 cells"""
    out = []
    for seed, side, free, layers, grid, nz, dz in ((31, 60, 5200, 6, 77, 61, 0.7), (32, 44, 2300, 5, 49, 45, 0.9),
                                                   (33, 72, 7100, 6, 95, 70, 0.61)):
        box = 2.0 * np.ceil(0.4 * side)
        out.append(configs.make_tissue(seed, nmx=side, nmy=side, lx=box, ly=box, nx=grid, ny=grid, nz=nz, n_fix=16,
                                       n_free=min(free, int(0.9 * (box / 2) ** 2 * layers)), n_layers=layers,
                                       dead_top=True, n_hot_alive=8, lz=nz * dz))
    return out


def run(specs, tuning, n_sub):
    from epi_amd import native
    ts = native.TissueSet([s["geometry"] for s in specs])
    ts.set_tuning(tuning)
    for t, s in enumerate(specs):
        ts.load(t, s)
    ts.setup_map_lat()
    zz = ts.calc_zzmax()
    ts.calc_ca2p_n(zz, n_sub)
    out = [(ts.get_cells(t), ts.get_fields(t)) for t in range(ts.T)]
    ts.close()
    return out, zz


def test_fused_runs_of_several_tissues():
    specs = tissues()
    ref, zz = run(specs, {}, 5)   # the defaults: fused, two planes a tile, XCD 1
    # the launch's workgroups: 16 cells past the membrane, or 128 points by 2 planes, each
    afm = sum(-(-(s["cells"]["x"].size + 64 - s["nmemb"] - s["nder"]) // 16) for s in specs)
    izb = [int((z + 2.8) / (s["geometry"].lz / s["geometry"].nz)) for s, z in zip(specs, zz)]
    tiles = sum(-(-s["geometry"].nx * s["geometry"].ny // 128) * -(-b // 2) for s, b in zip(specs, izb))
    assert afm % 8 and afm + tiles >= 2048
    for shape in ({"xcd": 0}, {"ca_group": 16}, {"atp_zb": 1}, {"ca_fuse": 0}):
        got, _ = run(specs, shape, 5)
        for t, (a, b) in enumerate(zip(got, ref)):
            for key in KEYS:
                assert np.array_equal(a[0][key], b[0][key]), (shape, t, key)
            for key in ("atp", "atp_next"):
                assert np.array_equal(a[1][key], b[1][key]), (shape, t, key)
    for t, s in enumerate(specs):
        (got,), _ = run([s], {}, 5)
        for key in KEYS:
            assert np.array_equal(got[0][key], ref[t][0][key]), (t, key)
        for key in ("atp", "atp_next"):
            assert np.array_equal(got[1][key], ref[t][1][key]), (t, key)
