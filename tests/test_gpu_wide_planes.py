"""A Ca solve on grids past the 32-bit limits: planes larger than 4 GB (64-bit
offsets in the ATP update, never fused) and more than 2^32 points in all (the
corners' words).  The same cells in a large box and in a small one, whose grid
spacing, and so every value near the cells, is the same."""
import ctypes as C

import numpy as np
import pytest

from epi_amd.configs import ALIVE, DEAD, FIX, MUSUME

from helpers import sheet_spec

pytestmark = pytest.mark.gpu

DX = 0.125
BYTES_PER_POINT = 42   # grid arrays of a context


def specs(seed, nx, ny, nz, lz, x0, y0, z0, n=60):
    """the tissue in a box of 160 x 160 points and, moved by (x0, y0), in one of nx x ny; multiples of
    2^-16, so that the move and the differences are exact"""
    r = np.random.default_rng(seed)
    q = lambda v: np.round(v * 65536) / 65536
    free = [dict(state=int(r.choice([ALIVE, ALIVE, DEAD, FIX, MUSUME])), x=float(q(r.uniform(4, 16))),
                 y=float(q(r.uniform(4, 16))), z=float(q(r.uniform(z0 - 1.5, z0))), agek=float(r.uniform(0, 6)))
            for _ in range(n)]
    out = []
    for size, dx, dy in (((160, 160, nz), 0.0, 0.0), ((nx, ny, nz), x0, y0)):
        s = sheet_spec(free, L=20.0, grid=(160, 160, nz), lz=lz)
        c, g = s["cells"], s["geometry"]
        g.nx, g.ny, g.lx, g.ly = size[0], size[1], size[0] * DX, size[1] * DX
        c["x"], c["y"] = q(c["x"]) + dx, q(c["y"]) + dy
        m = c["x"].size
        v = np.random.default_rng(seed + 1)
        s["values"] = {k: 0.1 + v.uniform(-0.05, 0.05, m) for k in ("ca2p", "ip3", "ca2p_avg")}
        s["values"]["ex_inert"] = np.full(m, 0.97)
        s["fields"] = None
        out.append(s)
    return out


def solves(spec, shapes, n_sub):
    """the cells after each of a row of solves of n_sub sub-steps, one per launch shape"""
    from epi_amd import native
    g = native.Tissue(spec["geometry"])
    g.set_params({"Da": 0.1})   # stable at this spacing
    g.load(spec)
    g.setup_map_lat()
    zz = g.calc_zzmax()
    out = []
    for shape in shapes:
        g.set.set_tuning(shape)
        g.set.calc_ca2p_n(zz, n_sub)
        out.append(g.get_cells())
    g.close()
    return out


def check(small, large, n_sub=6):
    """4 x 6 sub-steps: what differs, the boxes' seams 32 points from any cell, does not reach the cells"""
    shapes = [{"atp_zb": 1}, {"atp_zb": 2}, {"atp_zb": 8}, {"ca_fuse": 0, "atp_zb": 4}]
    refs = solves(small, [{}] * 4, n_sub)
    ip3 = refs[-1]["ip3"]
    assert np.all(np.isfinite(ip3)) and np.ptp(ip3) > 0 and np.ptp(refs[-1]["gj"]) > 0
    for shape, got, ref in zip(shapes, solves(large, shapes, n_sub), refs):
        for key in ("conn", "ca2p", "ca2p_next", "ip3", "ip3_next", "ca2p_avg", "ex_inert", "gj"):
            assert np.array_equal(got[key], ref[key]), (shape, key)


@pytest.mark.parametrize("nx,ny,nz,lz,y0,top", [
    (23200, 23200, 2, 10.0, 2878.0, 7.25),       # iz_bound = nz; the upper cells' rows lie past byte 2^32 of a plane
    (1600, 1616, 1680, 210.0, 0.0, 206.5),       # 4.4 G points; the upper cells' planes lie past point 2^32
])
def test_large_grids(nx, ny, nz, lz, y0, top):
    from epi_amd import native
    points = (nx + 16) // 16 * 16 * (ny + 1) * (nz + 1)
    free, total = C.c_size_t(), C.c_size_t()
    assert native.load_library().hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # found through its own HIP runtime
    if free.value < 1.05 * BYTES_PER_POINT * points:
        pytest.skip("not enough free memory on the card")
    check(*specs(3, nx, ny, nz, lz, 0.0, y0, top))


def gradient(spec, n_sub):
    from epi_amd import native
    g = native.Tissue(spec["geometry"])
    g.set_params({"Da": 0.1})
    g.load(spec)
    g.setup_map_lat()
    g.set.rd_begin(g.calc_zzmax())
    target = g.get_cells()["ca2p"] * 0.97
    loss, grads = g.set.rd_adjoint([dict(du=0.01, dp=0.1, gj0=0.99)], n_sub, n_sub, [target])
    g.close()
    return loss[0], grads[0]


def test_window_box_past_2_31_points():
    """the voxels that a cell owns in a window: 32 bits, unsigned"""
    from epi_amd import native
    nx, ny, nz, lz, top = 1600, 1616, 850, 106.25, 102.75   # iz_bound 844: the box holds 2.2 G points
    points = (nx + 16) // 16 * 16 * (ny + 1) * (nz + 1)
    free, total = C.c_size_t(), C.c_size_t()
    assert native.load_library().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    # the context, the window's snapshot and three adjoint grids, one checkpoint
    if free.value < 1.05 * (BYTES_PER_POINT + 56) * points:
        pytest.skip("not enough free memory on the card")
    small, large = specs(6, nx, ny, nz, lz, 0.0, 0.0, top)
    ref, got = gradient(small, 4), gradient(large, 4)
    assert ref[0] > 0 and got[0] == pytest.approx(ref[0], rel=1e-12)
    for k in ("du", "dp", "gj0"):     # FP64 atomics in another order
        assert got[1][k] == pytest.approx(ref[1][k], rel=1e-9), k
    assert np.allclose(got[1]["kpa"], ref[1]["kpa"], rtol=1e-9, atol=1e-9 * np.max(np.abs(ref[1]["kpa"])))
