"""The grid index arithmetic of the kernels, built for the host from the same
headers and run on sparse grids (CPU only): the eight grid_avg8 corners
(utils.h:18-23) of a cell in a Ca solve (ca_corner.h) against the seven-point
ATP update (ca2p.cpp:302-338) written out -- inside the grid, at its periodic
seams, at the mirrored bottom, the top plane and iz_bound -- and the voxel-map
stamp (field_step.h) against setup_map_lat's loops (map.cpp:39-166)."""
import ctypes as C
import itertools
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("grid") / "libgrid.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "native", "grid_index_check.cpp"), "-o", out], check=True)
    return C.CDLL(out)


def corners(lib, nx, ny, nz, izb, x, y, z, mask, seed):
    out, want = np.full(8, -1.0), np.full(8, -2.0)
    raw, raw_want = np.full(8, -1, np.int64), np.full(8, -2, np.int64)
    rc = lib.corner_check(nx, ny, nz, izb, x, y, z, mask, seed,
                          *(a.ctypes.data_as(C.c_void_p) for a in (out, want, raw, raw_want)))
    if rc:
        pytest.skip("no address space for the grid")
    # the two sides add the same dozen terms of order 1 in another order
    assert np.allclose(out, want, rtol=1e-13, atol=1e-14), (x, y, z, out, want)
    assert np.array_equal(raw, raw_want), (x, y, z)


@pytest.mark.parametrize("nx,ny,nz,izb", [(5, 7, 6, 4), (2, 3, 2, 2), (33, 16, 9, 9), (15, 15, 4, 1), (16, 31, 3, 0)])
@pytest.mark.parametrize("mask", [1, 2])
def test_every_corner_of_small_grids(lib, nx, ny, nz, izb, mask):
    at = lambda n: sorted({0, 1, n // 2, n - 2, n - 1})
    for i, (x, y, z) in enumerate(itertools.product(at(nx), at(ny), at(nz))):
        corners(lib, nx, ny, nz, izb, x, y, z, mask, i)


@pytest.mark.parametrize("nx,ny,nz,izb", [
    (1600, 1600, 1680, 1680),    # 4.35 G points in planes of 21 MB
    (23200, 23200, 8, 8),        # 4.85 G points in planes of 4.3 GB
    (1040, 1040, 8100, 4000),    # 8.9 G points, the top half above iz_bound
])
def test_corners_of_grids_past_32_bit_indices(lib, nx, ny, nz, izb):
    first = (1 << 32) // ((nx + 1 + 15) // 16 * 16 * (ny + 1))   # the plane that holds point 2^32
    for i, (x, y, z) in enumerate(itertools.product((0, nx - 1), (0, ny // 2, ny - 1),
                                                    {1, first - 1, first, first + 1, nz - 2, nz - 1})):
        if z < nz:
            corners(lib, nx, ny, nz, izb, x, y, z, 1, i)


@pytest.mark.parametrize("nx,ny,nz,lx,ly,lz", [
    (16, 20, 12, 12.8, 14.0, 10.0),
    (46400, 46400, 2, 5800.0, 5800.0, 10.0),   # a plane of 2.15 G points: row offsets past 2^31
])
@pytest.mark.parametrize("lanes", [1, 4, 16])
def test_stamp(lib, nx, ny, nz, lx, ly, lz, lanes):
    from epi_amd.configs import ALIVE, DEAD, FIX, MEMB
    x = [1.0, 0.01, lx - 0.01, 3.3, lx / 2, 2.2]
    y = [1.0, 0.02, ly - 0.03, ly - 0.6, ly - 1.9, ly / 2]
    z = [lz / 2 + 0.1] * len(x)
    state = np.array([MEMB, ALIVE, DEAD, FIX, ALIVE, MEMB], np.uint8)
    xs, ys, zs = (np.array(a, np.float64) for a in (x, y, z))
    r = np.full(len(x), 1.4)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    lib.stamp_check.restype = C.c_longlong
    bad = lib.stamp_check(nx, ny, nz, C.c_double(lx), C.c_double(ly), C.c_double(lz), len(x), p(xs), p(ys), p(zs), p(r),
                          p(state), lanes)
    if bad < 0:
        pytest.skip("no address space for the grid")
    assert bad == 0
