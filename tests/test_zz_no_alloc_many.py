"""epi_calc_ext_stim_noalloc with as many grids as its set-up block has lanes,
more, and the most it takes: every grid's B equals the call with that grid
alone (which test_zz_no_alloc compares with calc_ext_stim), a grid whose
iz_bound lies outside [0, nz] is left as it was and gets its code."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import Hip, View

pytestmark = pytest.mark.gpu

SHAPES = [(7, 6, 9), (16, 17, 8), (5, 5, 30)]   # nx, ny, nz
OUT_OF_GRID = 4


def put_inputs(hip, seed):
    """per shape: a view without its output, and the output's start values"""
    r = np.random.default_rng(seed)
    made = []
    for nx, ny, nz in SHAPES:
        xp, pl = nx + 2, (nx + 2) * (ny + 1) + 5
        n = pl * (nz + 1)
        v = View()
        v.nx, v.ny, v.nz, v.xp, v.pl, v.lz = nx, ny, nz, xp, pl, nz * 0.8
        v.zzmax = 0.8 * (nz - 2.5) - 2.8
        v.b_in = hip.put(r.uniform(0, 1, n))
        v.cmap1 = hip.put(r.integers(-1, 40, n).astype(np.int32))
        v.cmap2 = hip.put(r.integers(0, 2, n).astype(np.uint8))
        v.state = hip.put(r.choice([0, 1, 3, 5], 40).astype(np.uint8))
        v.agek = hip.put(r.uniform(20, 40, 40))
        made.append((v, r.uniform(0, 1, n)))
    return made


def sweep(hip, lib, views, n):
    d_views = hip.put(np.frombuffer(bytes(views), dtype=np.uint8))
    d_err = hip.put(np.full(n, -1, dtype=np.int32))
    assert lib.epi_calc_ext_stim_noalloc(C.c_void_p(d_views), n, C.c_void_p(d_err), None) == 0
    hip.sync()
    return hip.get(d_err, n, np.int32)


@pytest.mark.parametrize("n", [1, 63, 256, 257, 1023, 1024])
def test_many_grids(n):
    from epi_amd import native
    lib = native.load_library()
    lib.epi_calc_ext_stim_noalloc.argtypes = [C.c_void_p, C.c_int32, C.c_void_p, C.c_void_p]
    hip = Hip()
    try:
        print(f"no-alloc sweep of {n} grids", flush=True)
        made = put_inputs(hip, 5)
        alone = []
        for v, start in made:
            one = (View * 1)()
            C.memmove(one, C.byref(v), C.sizeof(View))
            one[0].b_out = hip.put(start)
            assert list(sweep(hip, lib, one, 1)) == [0]
            alone.append(hip.get(one[0].b_out, start.size, np.float64))
            assert not np.array_equal(alone[-1], start)
        views = (View * n)()
        bad = np.array([i % 5 == 4 for i in range(n)])
        kinds = [i % len(SHAPES) for i in range(n)]
        at = np.concatenate([[0], np.cumsum([made[k][1].size for k in kinds])]).astype(int)
        out = hip.put(np.concatenate([made[k][1] for k in kinds]))
        for i, k in enumerate(kinds):
            C.memmove(C.byref(views, i * C.sizeof(View)), C.byref(made[k][0]), C.sizeof(View))
            views[i].b_out = out + 8 * int(at[i])
            if bad[i]:
                views[i].zzmax = 1e3 if i % 2 else -1e3
        err = sweep(hip, lib, views, n)
        assert np.array_equal(err, np.where(bad, OUT_OF_GRID, 0))
        got = hip.get(out, int(at[-1]), np.float64)
        for i, k in enumerate(kinds):
            want = made[k][1] if bad[i] else alone[k]
            assert np.array_equal(got[at[i]:at[i + 1]], want), (i, k)
    finally:
        hip.free()
