"""The mechanics window's gradient on tissues that mix every cell state, so that
an entry of a row is planned for its handler, for the other cell, for both (a
DER-DER pair) or for none, with division partners inside and outside each
other's list, against the oracle's reverse pass.  Tolerances as for the other
gradients: FP64 sums in another order, 1e-8."""
import numpy as np
import pytest

from test_gpu_force_laws import mixed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed,pitch,der_layers", [(1, 2.0, 1), (2, 2.3, 2), (3, 2.0, 0), (4, 2.1, 3)])
@pytest.mark.parametrize("n_steps,every", [(1, 1), (5, 2)])
def test_mixed_states(oracle_mod, seed, pitch, der_layers, n_steps, every):
    from epi_amd import native
    spec = mixed(seed, pitch, der_layers)
    gt, ot = native.Tissue(spec["geometry"]), oracle_mod.OracleTissue(spec["geometry"])
    for t in (gt, ot):
        t.load(spec)
        t.connect_cell()
    base = dict(eps=0.01, k_adh=3.0, k_spring=25.0, k_bend=0.5)
    tgt = ot.mech_forward(n_steps, eps=0.0105, k_adh=3.15, k_spring=26.25, k_bend=0.525)
    tgt = tgt + 0.01 * np.random.default_rng(seed).uniform(-1, 1, tgt.shape)
    lo, go = ot.mech_adjoint(n_steps, tgt, **base)
    print(f"mech plan: seed {seed}, {der_layers} DER layers, {n_steps} steps", flush=True)
    gt.set.mech_begin()
    loss, grads = gt.set.mech_adjoint([base], n_steps, every, [tgt])
    gt.set.mech_end()
    assert loss[0] == pytest.approx(lo, rel=1e-12)
    for k in go:
        assert grads[0][k] == pytest.approx(go[k], rel=1e-8), k
    gt.close()
