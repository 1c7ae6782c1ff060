"""The mixed operator's window format (columns as slots of the row's 27-cell
window, staged in LDS per tile of rows) against the FP64 path's own formats on
the same particles: tiles that fill one pass, tiles that are halved because
their cells do not fit, periodic boxes of the least size, windows that do not
fit the 11-bit slots, and one, two and four lanes per row."""
from __future__ import annotations

import numpy as np
import pytest

from fluidized_bed_master_amd import abi, configs

pytestmark = pytest.mark.gpu


def _assembled(p, parts, prec):
    from fluidized_bed_master_amd.sophia import Sophia
    g = Sophia(p, parts, precision=prec)
    g.nnps(); g.prep(); g.interaction(); g.dem_interaction(); g.sph_dem_coupling(); g.predict()
    mixed = prec == abi.PREC_MIXED
    g.ppe(abi.ppe_opts(method=abi.PPE_BICGSTAB, precision=abi.PPE_MIXED_IR if mixed else abi.PPE_FP64, rtol=1e-4,
                       zero_mean=1 if p.periodic_mask else 0))
    return g


def _sparse():
    # a thin sheet of fluid in a tall, wide domain: most cells are empty, so 256
    # consecutive particles span far more planes than one tile holds
    p, parts = configs.isph_dem_column(60, 60, 2, 1.0e-3, wall_layers=1, tank_extra=14, jitter=0.02, seed=3)
    keep = (parts["p_type"] == abi.PT_FLUID) | (configs.uniform(9, len(parts)) < 0.2)
    return p, parts[keep]


def _overfull():
    # every particle four times, a little apart: windows of more than 2047
    p, parts = configs.taylor_green(12, jitter=0.05)
    more = np.concatenate([parts] * 4)
    for k, c in enumerate("xyz"):
        more[c] = np.mod(more[c] + configs.uniform(20 + k, len(more), 0.0, 0.02), 2 * np.pi)
    p.sph_max_neighbors = 480
    return p, more


CASES = {
    "column_4_lanes": (lambda: configs.small_isph_dem(seed=7), 0),
    "column_2_lanes": (lambda: configs.isph_dem_column(41, 37, 33, 1.0e-3, jitter=0.05, seed=4, u_noise=0.01), 0),
    "sparse_halved_tiles": (_sparse, 0),
    "box_three_cells": (lambda: configs.taylor_green(9, jitter=0.05), 0),
    "box_1_lane": (lambda: configs.taylor_green(80, jitter=0.05), 0),
    "box_drifted_2_lanes": (lambda: configs.taylor_green(37, jitter=0.05, drift=(0.3, 0.2, 0.1)), 0),
    "overfull_windows": (_overfull, 4),
}


@pytest.mark.parametrize("name", CASES)
def test_window_operator_matches_fp64_formats(name):
    """y = A x: hi + lo (FP64 sums) within the FP32 geometry's rounding of the
    coefficients, 2^-20 of sum_j |a_ij| |x_i - x_j| <= 2 d_i max |x|, and the
    inner operator within its 16-bit significands besides (2^-16)."""
    make, index_bytes = CASES[name]
    p, parts = make()
    a, b = _assembled(p, parts, abi.PREC_MIXED), _assembled(p, parts, abi.PREC_FP64)
    assert a.ppe_layout()["index_bytes"] == index_bytes
    assert a.ppe_layout()["nnz"] == b.ppe_layout()["nnz"]
    d, _, rows = b.get_ppe_system()
    r = rows == 1
    assert np.array_equal(a.get_ppe_system()[2], rows) and r.sum() > 0
    x = np.random.default_rng(5).uniform(-1, 1, len(rows)) * r
    ref = b.ppe_apply(x)
    scale = np.maximum(2 * np.abs(d[r]), 1e-3 * np.abs(d[r]).max())
    e = np.abs(a.ppe_apply(x) - ref)[r] / scale
    assert e.max() <= 2.0 ** -18, (name, e.max())
    if index_bytes == 0:
        e = np.abs(a.matvec_probe(0, x, reps=1)[0] - ref)[r] / scale
        assert e.max() <= 2.0 ** -16 + 2.0 ** -18, (name, e.max())
    a.close()
    b.close()
