"""Gradient of the learned warm start where a particle's neighbour list does not
fit one gathered buffer of 128 edges, and where lists end inside a tile of 16 or a
gather of 64."""
import ctypes as C

import numpy as np
import pytest

from fluidized_bed_master_amd import abi, configs, learned
from oracle import mlp
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_MIXED])
@pytest.mark.parametrize("h_scale,longest", [(0.8, (16, 64)), (1.25, (129, 256))])
def test_gradient_over_list_lengths(h_scale, longest, prec):
    from fluidized_bed_master_amd.sophia import Sophia
    p, parts = configs.small_isph_dem(n=9, nz=10, seed=7)
    parts["h"] *= h_scale
    g = Sophia(p, parts, precision=prec)
    for f in (g.nnps, g.prep, g.interaction, g.dem_interaction, g.sph_dem_coupling, g.predict):
        f()
    g.ppe(abi.ppe_opts(method=abi.PPE_JACOBI))
    w = learned.init_params(seed=12, out_scale=1.0)
    w[mlp.OFF_B1:mlp.OFF_W2] = 0.3 * learned.normal(3, mlp.OFF_W2 - mlp.OFF_B1)
    w[mlp.OFF_B2:mlp.OFF_W3] = 0.3 * learned.normal(4, mlp.OFF_W3 - mlp.OFF_B2)
    g.mlp_set_params(w)
    s1, _, _ = g.get_particles(abi.SPH)
    X, h, pprev = np.stack([s1["x"], s1["y"], s1["z"]], 1), s1["h"], s1["pres"].copy()
    nf, scale = np.zeros(len(X) * 2, np.float32), C.c_double()
    abi.check(g.lib.sophia_mlp_features(g._ctx, abi.ptr(nf), len(X), C.byref(scale)), "features")
    _, _, rows = g.get_ppe_system()
    src, dst = mlp.edges(X, h, p.kappa)
    m = rows.astype(bool)
    assert longest[0] <= np.bincount(src, minlength=len(X))[m].max() <= longest[1]
    # one-signed errors: a gradient entry is then a sum of terms mostly of one sign
    t_norm = 3.0 + np.random.default_rng(1).normal(0, 0.3, len(X))
    loss, grad = g.mlp_loss_grad(pprev + scale.value * t_norm)
    loss_ref, ref, _ = mlp.loss_grad(w, X, h, nf.reshape(-1, 2).astype(np.float64), rows, src, dst, t_norm, bf=True)
    # The kernel rounds dZ2 and dZ1 to BF16 for the products (2^-9 a term each) and
    # a ReLU within rounding of 0 may switch, on top of what the oracle rounds:
    # 2 * 2^-9 * sum|t| / |sum t|, with the ratio at most 7 for one-signed errors.
    # (With errors of both signs the ratio grows as the square root of the rows: 30
    # here, and W1 differs by 4 % of what is left of its sum.)
    assert abs(loss - loss_ref) / loss_ref < 2e-3, (loss, loss_ref)
    blocks = [mlp.OFF_W1, mlp.OFF_B1, mlp.OFF_W2, mlp.OFF_B2, mlp.OFF_W3, mlp.OFF_B3, mlp.OFF_W4, mlp.OFF_B4,
              mlp.NPARAM]
    for a, b in zip(blocks, blocks[1:]):
        assert rel_err(grad[a:b], ref[a:b]) < 3e-2, (a, rel_err(grad[a:b], ref[a:b]))


def test_gradient_sums_round_once_in_a_thousandth_of_the_rows():
    """Equal errors on all rows and messages that are whole multiples of b2: every
    term of dW3 is known, and what its entries differ by from w4_l b2_k is the
    rounding of the FP32 accumulators, at most rows / 1024 additions each.  An
    addition rounds by up to 2^-25 of a partial sum that grows linearly, N 2^-25 of
    the whole sum if all round one way; three quarters of that here (half is what is
    seen, 9.3e-7, and 1.85e-6 where an accumulator takes twice as many)."""
    from fluidized_bed_master_amd.sophia import Sophia
    p, parts = configs.isph_dem_column(40, 40, 40, 1.0e-3, seed=2)
    w = np.zeros(mlp.NPARAM, np.float32)
    b2, w4 = 0.5 + np.arange(64) / 128, 1.0 + np.arange(64) / 64  # exact in BF16
    w[mlp.OFF_B2:mlp.OFF_W3], w[mlp.OFF_B3:mlp.OFF_W4], w[mlp.OFF_W4:mlp.OFF_B4] = b2, 1.0, w4
    with Sophia(p, parts, precision=abi.PREC_FP64) as g:
        for f in (g.nnps, g.prep, g.interaction, g.dem_interaction, g.sph_dem_coupling, g.predict):
            f()
        g.ppe(abi.ppe_opts(method=abi.PPE_JACOBI))
        g.mlp_set_params(w)
        pprev = g.get_particles(abi.SPH)[0]["pres"].copy()
        nf, scale = np.zeros(len(pprev) * 2, np.float32), C.c_double()
        abi.check(g.lib.sophia_mlp_features(g._ctx, abi.ptr(nf), len(pprev), C.byref(scale)), "features")
        rows = (g.get_ppe_system()[2] == 1).sum()
        assert rows == 64000
        for err in (0.1, 0.7, 2.3):
            _, grad = g.mlp_loss_grad(pprev + scale.value * (w4.sum() - err))
            q = grad[mlp.OFF_W3:mlp.OFF_B3].reshape(64, 64) / np.outer(w4, b2)
            assert np.abs(q / np.median(q) - 1).max() <= 0.75 * rows / 1024 * 2.0 ** -25
