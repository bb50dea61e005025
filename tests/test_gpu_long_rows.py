"""Forces over lists that the caller sets (epi_set_lists) and that are longer than
any the library has built: rows past the first LDS size (40 entries), past the
last (64), and short ones, in one step and in a window with its gradient,
against the oracle's serial loop."""
import numpy as np
import pytest

from epi_amd.configs import ALIVE, DEAD, MUSUME

from helpers import pdiff, sheet_spec

pytestmark = pytest.mark.gpu

L = 16.0


def tissue(seed):
    r = np.random.default_rng(seed)
    free = [dict(state=int(r.choice([ALIVE, ALIVE, DEAD, MUSUME])), agek=float(r.choice([1.0, 3.5])),
                 x=float((k % 8 + 0.5) * 2 + r.uniform(-0.1, 0.1)), y=float((k // 8 % 8 + 0.5) * 2 + r.uniform(-0.1, 0.1)),
                 z=float(2.9 + 2.0 * (k // 64) + r.uniform(-0.1, 0.1))) for k in range(192)]
    spec = sheet_spec(free, nmx=16, nmy=16, L=L, grid=(16, 16, 24), lz=24.0)
    spec["cells"]["z"][:spec["nmemb"]] += r.uniform(-0.05, 0.05, spec["nmemb"])
    return spec


def longer(cells, m, want):
    """the tissue's lists with further mutual pairs, nearest first, until a free cell has want(i) entries"""
    n = cells["n"]
    rows = [list(cells["conn"][cells["conn_ptr"][i]:cells["conn_ptr"][i + 1]]) for i in range(n)]
    p = [cells[k][m:] for k in "xyz"]
    d = pdiff(p[0][:, None], p[0][None], L) ** 2 + pdiff(p[1][:, None], p[1][None], L) ** 2 + (p[2][:, None] - p[2]) ** 2
    for i in range(n - m):
        for j in np.argsort(d[i], kind="stable")[1:]:
            if len(rows[m + i]) >= want(i):
                break
            if m + j not in rows[m + i]:
                rows[m + i].append(m + int(j))
                rows[m + j].append(m + i)
    for i in range(m, n):   # canonical order: lower partners, then the others ascending
        rows[i] = sorted(rows[i])
    ptr = np.concatenate([[0], np.cumsum([len(x) for x in rows])]).astype(np.int32)
    return ptr, np.concatenate([np.asarray(x, np.int32) for x in rows]), max(len(x) for x in rows)


@pytest.mark.parametrize("want,lo,hi", [(lambda i: 41, 41, 64), (lambda i: 75 if i == 5 else 20, 65, 200)])
def test_rows_that_the_caller_sets(oracle_mod, want, lo, hi):
    from epi_amd import native
    spec = tissue(2)
    g, o = native.Tissue(spec["geometry"]), oracle_mod.OracleTissue(spec["geometry"])
    for t in (g, o):
        t.load(spec)
    ptr, conn, longest = longer(o.get_cells(), spec["nmemb"], want)
    assert lo <= longest <= hi
    for t in (g, o):
        t.set_lists(ptr, conn)
        t.cell_interaction()
        t.pos_copy()
    a, b = g.get_cells(), o.get_cells()
    assert g.error() == o.error() == 0
    for k in "xyz":
        assert np.array_equal(a[k], b[k]), (k, int(np.count_nonzero(a[k] != b[k])))
    base = dict(eps=0.01, k_adh=3.0, k_spring=25.0, k_bend=0.5)
    tgt = o.mech_forward(4, eps=0.0105, k_adh=3.15, k_spring=26.25, k_bend=0.525)
    tgt = tgt + 0.01 * np.random.default_rng(3).uniform(-1, 1, tgt.shape)
    lo_, go = o.mech_adjoint(4, tgt, **base)
    g.set.mech_begin()
    loss, grads = g.set.mech_adjoint([base], 4, 2, [tgt])
    g.set.mech_end()
    # FP64 sums in another order, as in the other gradient tests
    assert loss[0] == pytest.approx(lo_, rel=1e-12)
    for k in go:
        assert grads[0][k] == pytest.approx(go[k], rel=1e-8), k
    g.close()
