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
    coefficients, and the inner operator within its 16-bit significands besides
    (2^-16), of sum_j |a_ij| |x_i - x_j| <= 2 d_i max |x|.  That rounding is 2^-22 of a
    coefficient and more where it goes to 0 as (1 - q)^3: 2^-22 of the sum at most in
    columns, 2^-19 in one of the largest box's 512,000 rows, and twice that is asked.
    Rows with less than a thousandth of the largest diagonal have only such
    coefficients (a spray's 2^-14) and are held to that thousandth."""
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


def _column(more=None, **kw):
    # walls 14 layers above the surface, and `more` records in the freeboard
    p, parts = configs.isph_dem_column(12, 12, 12, 1.0e-3, tank_extra=14, jitter=0.02, seed=3, u_noise=0.01, **kw)
    if more is None:
        return p, parts
    extra = parts[parts["p_type"] == abi.PT_FLUID][:len(more)].copy()
    extra["pres"] = 0.0
    for k, fields in enumerate(more):
        for f, v in fields.items():
            extra[f][k] = v
    return p, np.concatenate([parts, extra])


def _sphere_above_surface():
    # wall particles within reach of the sphere and of no fluid: eps = -1e18, and
    # eps rho is beyond FP32
    p, parts = _column(d_dem=2.0e-3, dem_height=3.0e-3, max_dem=1)
    s = parts["p_type"] == abi.PT_DEM
    assert s.sum() == 1
    for c, v in zip("xyz", (1.2e-3, 6.0e-3, 17.0e-3)):
        parts[c][s] = v
    return p, parts


def _dummy_without_density():
    # i_type 3: in no cell and in no sum
    return _column([{"x": 6e-3, "y": 6e-3, "z": 18.5e-3, "i_type": 3, "rho": 0.0}])


def _heavy_stranger():
    # one row 2^40 denser than the others and with no neighbour: every other row
    # takes its range from its own coefficients
    p, parts = _column([{"x": 6e-3, "y": 6e-3, "z": 18.5e-3, "p_type": 2}])
    p.rho_water = 1000.0 * 2.0 ** 40
    return p, parts


@pytest.mark.parametrize("make", [_sphere_above_surface, _dummy_without_density, _heavy_stranger])
def test_particles_that_no_row_couples_to_leave_the_operator_alone(make):
    """The product and a converged solve beside the FP64 path's, with the bounds
    of the test above for rows, each on its own diagonal."""
    p, parts = make()
    a, b = _assembled(p, parts, abi.PREC_MIXED), _assembled(p, parts, abi.PREC_FP64)
    assert a.ppe_layout()["index_bytes"] == 0
    d, _, rows = b.get_ppe_system()
    r = (rows == 1) & (d != 0)
    x = np.random.default_rng(5).uniform(-1, 1, len(rows)) * r
    ref = b.ppe_apply(x)
    scale = 2 * np.abs(d[r])
    assert (np.abs(a.ppe_apply(x) - ref)[r] / scale).max() <= 2.0 ** -18
    assert (np.abs(a.matvec_probe(0, x, reps=1)[0] - ref)[r] / scale).max() <= 2.0 ** -16 + 2.0 ** -18
    a.close()
    b.close()
    from fluidized_bed_master_amd.sophia import Sophia
    pres = []
    for prec in (abi.PREC_MIXED, abi.PREC_FP64):
        mixed = prec == abi.PREC_MIXED
        with Sophia(p, parts, precision=prec) as g:
            st = g.step(abi.ppe_opts(method=abi.PPE_BICGSTAB, rtol=1e-8,
                                     precision=abi.PPE_MIXED_IR if mixed else abi.PPE_FP64))
            assert st["converged"], st
            s1 = g.get_particles(abi.SPH)[0]
            pres.append(s1["pres"][s1["p_type"] == abi.PT_FLUID])
    assert np.abs(pres[0] - pres[1]).max() <= 1e-5 * np.abs(pres[1]).max()


def test_row_far_below_the_others_keeps_its_precision():
    """Two particles alone, 0.9995 of the support apart: coefficients 2^-34 of the
    column's.  With hi + lo at 2^-40 of the coefficient and an inner diagonal that
    takes up hi's rounding in FP32, A 1 = 0 to 2^-40 and 2^-23 of the diagonal."""
    h = 1.3e-3
    p, parts = _column([{"x": 4.7e-3, "y": 6e-3, "z": 18.5e-3},
                        {"x": 4.7e-3 + 0.9995 * 2 * h, "y": 6e-3, "z": 18.5e-3}])
    a = _assembled(p, parts, abi.PREC_MIXED)
    assert a.ppe_layout()["index_bytes"] == 0
    d, _, rows = a.get_ppe_system()
    s1 = a.get_particles(abi.SPH)[0]
    pair = (s1["p_type"] == abi.PT_FLUID) & (s1["z"] > 18e-3)
    assert pair.sum() == 2 and (rows[pair] == 1).all()
    assert (d[pair] > 0).all() and d[pair].max() < 2.0 ** -33 * np.median(d[rows == 1])
    one = (rows == 1).astype(float)
    assert (np.abs(a.ppe_apply(one))[pair] <= 2.0 ** -39 * d[pair]).all()
    assert (np.abs(a.matvec_probe(0, one, reps=1)[0])[pair] <= 2.0 ** -22 * d[pair]).all()
    # the coupling itself, to its 16-bit significand
    e = np.zeros(len(rows))
    i, j = np.flatnonzero(pair)
    e[j] = 1.0
    assert abs(a.ppe_apply(e)[i] + d[i]) <= 2.0 ** -39 * d[i]
    assert abs(a.matvec_probe(0, e, reps=1)[0][i] + d[i]) <= 2.0 ** -16 * d[i]
    a.close()


def _film():
    # two layers of fluid in a tray with sparse walls: in the upper cells of the
    # walls a run of planes holds a handful of particles
    p, parts = configs.isph_dem_column(300, 300, 2, 1.0e-3, jitter=0.02, seed=3, tank_extra=10)
    keep = (parts["p_type"] == abi.PT_FLUID) | (configs.uniform(9, len(parts)) < 0.3)
    return p, parts[keep]


def _wide(nx=40, ny=40, nz=40):
    # a column in one corner of a domain sixteen times as wide: the cells of one
    # x-row end and those of the next begin 200 apart
    p, parts = configs.isph_dem_column(nx, ny, nz, 1.0e-3, jitter=0.02, seed=3)
    far = parts[:200].copy()
    far["x"] += 0.6
    return p, np.concatenate([far, parts])


def _spray(n=60, fill=0.02):
    # drops: single particles and small groups, most cells empty
    p, parts = configs.isph_dem_column(n, n, n, 1.0e-3, jitter=0.4, seed=3, wall_layers=1, u_noise=0.01)
    fluid = parts["p_type"] == abi.PT_FLUID
    u = configs.uniform(12, len(parts))
    drop = configs.uniform(13, (n // 4 + 1) ** 3) < fill  # groups of up to 4^3
    g = [np.minimum((parts[c] / 4e-3).astype(int), n // 4) for c in "xyz"]
    in_drop = drop[np.clip(g[0] + (n // 4 + 1) * (g[1] + (n // 4 + 1) * g[2]), 0, len(drop) - 1)]
    return p, parts[~fluid | (u < fill) | (fluid & in_drop & (u < 0.5))]


def _dense():
    # 1,000 particles and more around a cell: a tile's planes hold more than it stages
    p, parts = configs.taylor_green(22, jitter=0.05)
    more = np.concatenate([parts] * 2)
    for k, c in enumerate("xyz"):
        more[c] = np.mod(more[c] + configs.uniform(20 + k, len(more), 0.0, 0.1), 2 * np.pi)
    p.sph_max_neighbors = 240
    return p, more


def _freeboard():
    # walls three times the column's height: tiles of thin wall rings
    return configs.isph_dem_column(40, 42, 30, 1.0e-3, jitter=0.02, seed=3, tank_extra=90)


def _surface():
    # the top layer half in one cell layer and half in the next: a third of its rows
    # lie by ones and twos
    return configs.isph_dem_column(120, 120, 5, 1.0e-3, jitter=0.45, seed=3, tank_extra=6)


# (system, bytes per column index: 0 window slots, 4 where the rows lie thinly)
GAPS = {
    "film": (_film, 4),
    "wide": (_wide, 0),
    "wide_2_lanes": (lambda: _wide(60, 62, 70), 0),
    "freeboard": (_freeboard, 0),
    "surface": (_surface, 0),
    "spray": (_spray, 4),
    "spray_of_groups": (lambda: _spray(40, 0.3), 0),
    "dense": (_dense, 0),
}


@pytest.mark.parametrize("name", GAPS)
def test_tiles_with_gaps_match_fp64_formats(name):
    """Tiles planned around their rows' cells alone, and the u32 columns of thin
    systems: the product, the inner product and (two-level) the coarse operator
    beside the FP64 path's formats; a second assembly gives the same bits."""
    make, index_bytes = GAPS[name]
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
    assert (np.abs(a.ppe_apply(x) - ref)[r] / scale).max() <= 2.0 ** -18
    inner = a.matvec_probe(0, x, reps=1)[0]
    assert (np.abs(inner - ref)[r] / scale).max() <= 2.0 ** -16 + 2.0 ** -18
    full = a.ppe_apply(x)
    a.ppe(abi.ppe_opts(method=abi.PPE_BICGSTAB, precision=abi.PPE_MIXED_IR, max_iter=1,
                       zero_mean=1 if p.periodic_mask else 0))
    assert a.ppe_layout()["index_bytes"] == index_bytes
    assert np.array_equal(a.ppe_apply(x), full) and np.array_equal(a.matvec_probe(0, x, reps=1)[0], inner)
    if not p.periodic_mask:
        E = []
        for g, mixed in ((a, True), (b, False)):
            st = g.ppe(abi.ppe_opts(method=abi.PPE_BICGSTAB, rtol=1e-3, precond=abi.PRECOND_TWO_LEVEL, max_iter=200,
                                    guess=abi.GUESS_ZERO, precision=abi.PPE_MIXED_IR if mixed else abi.PPE_FP64))
            if st["precond_used"] == abi.PRECOND_TWO_LEVEL:
                E.append(g.ppe_coarse()[1].astype(float))
        assert len(E) == (0 if name == "spray" else 2)  # lone drops: a singular coarse operator
        # FP32 entries of sums of coefficients with relative errors of 2^-18
        if E:
            assert np.abs(E[0] - E[1]).max() <= 2.0 ** -17 * np.abs(E[1]).max()
    a.close()
    b.close()


@pytest.mark.parametrize("gaps,full,index_bytes,most", [
    (_wide, lambda: configs.isph_dem_column(40, 40, 40, 1.0e-3, jitter=0.02, seed=3), 0, 1.7),
    (_film, configs.c4_train, 4, 2.0)], ids=["wide", "film"])
def test_wall_cells_and_gaps_cost_no_tiles(gaps, full, index_bytes, most):
    """A pass over the wide domain takes little longer than one over its column alone
    (1.1 of it; 2.7 where every gap halves its tile until the planes fit), and one over
    the film no longer than over a full column of as many particles (0.8; 3.9)."""
    us = []
    for k, (p, parts) in enumerate((gaps(), full())):
        g = _assembled(p, parts, abi.PREC_MIXED)
        assert g.ppe_layout()["index_bytes"] == (index_bytes if k == 0 else 0)
        x = np.ones(len(g.get_ppe_system()[2]))
        us.append(min(g.matvec_probe(0, x, reps=50)[1] for _ in range(5)))
        g.close()
    assert us[0] <= most * us[1], us


@pytest.mark.parametrize("n", [17, 26, 40], ids=["even", "odd", "odd_drifted"])
def test_coarse_operator_across_a_periodic_wrap(n):
    """A box periodic along x with open sides (free-surface rows): the coarse
    operator of the window rows beside the FP64 path's, with an even and an odd number
    of aggregates along the period.  Couplings across the wrap belong to no pair of
    neighbouring aggregates and leave E; those of an odd number's last and first
    aggregate must not land in the diagonal."""
    p, parts = configs.taylor_green(n, jitter=0.05, drift=(0.3, 0.0, 0.0) if n == 40 else (0.0, 0.0, 0.0))
    p.periodic_mask = 1
    p.free_surface = 1
    for c in (1, 2):
        p.domain_max[c] = 0.96 * p.domain_max[c]
    parts = parts[(parts["y"] < 0.9 * 2 * np.pi) & (parts["z"] < 0.9 * 2 * np.pi)]
    E = []
    for prec in (abi.PREC_MIXED, abi.PREC_FP64):
        from fluidized_bed_master_amd.sophia import Sophia
        mixed = prec == abi.PREC_MIXED
        with Sophia(p, parts, precision=prec) as g:
            st = g.step(abi.ppe_opts(method=abi.PPE_BICGSTAB, rtol=1e-6, precond=abi.PRECOND_TWO_LEVEL,
                                     precision=abi.PPE_MIXED_IR if mixed else abi.PPE_FP64))
            assert st["converged"] and st["precond_used"] == abi.PRECOND_TWO_LEVEL, st
            dims, e, _ = g.ppe_coarse()
            assert dims[0] % 2 == (0 if n == 17 else 1) and dims[0] > 1, dims
            assert g.ppe_layout()["index_bytes"] == (0 if mixed else 4)
            E.append(e.astype(float))
    # FP32 entries of sums of coefficients with relative errors of 2^-18
    assert np.abs(E[0] - E[1]).max() <= 2.0 ** -17 * np.abs(E[1]).max()


def test_long_periodic_box_takes_u32_columns():
    """More than 1000 cells along a period: the records' ten bits no longer tell the
    images apart, so the columns are plain indices; the probe of the window operator
    is refused there."""
    p, parts = configs.taylor_green(4, jitter=0.05)
    dx, nx = 2 * np.pi / 4, 2880
    cut = np.concatenate([parts] * (nx // 4))
    cut["x"] = parts["x"].repeat(nx // 4) % (2 * np.pi) + 2 * np.pi * np.tile(np.arange(nx // 4), len(parts))
    for c in "yz":
        cut[c] = parts[c].repeat(nx // 4)
    cut["uy"] = 0.01 * np.sin(cut["x"])
    p.periodic_mask = 1
    p.free_surface = 1
    p.domain_max[0] = nx * dx
    a, b = _assembled(p, cut, abi.PREC_MIXED), _assembled(p, cut, abi.PREC_FP64)
    assert a.domain.NI > 1000
    assert a.ppe_layout()["index_bytes"] == 4 and a.ppe_layout()["nnz"] == b.ppe_layout()["nnz"]
    d, _, rows = b.get_ppe_system()
    r = rows == 1
    assert np.array_equal(a.get_ppe_system()[2], rows) and r.sum() > 1000
    x = np.random.default_rng(5).uniform(-1, 1, len(rows)) * r
    scale = np.maximum(2 * np.abs(d[r]), 1e-3 * np.abs(d[r]).max())
    # the record grid is a 1024th of the period here, 1.1 cells
    assert (np.abs(a.ppe_apply(x) - b.ppe_apply(x))[r] / scale).max() <= 2.0 ** -14
    with pytest.raises(abi.SophiaError):
        a.matvec_probe(0, x, reps=1)
    a.close()
    b.close()
