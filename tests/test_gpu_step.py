"""The one-launch level step (k_godunov_step) at the sizes where its boundary pieces and strips can
go wrong: domains of a few cells (no interior at all), bands that end in pieces of one cell, pieces
of exactly 23 cells, boxes whose edges cut the bands, free surfaces; and the strip height a launch
takes when none was set.

Slip weakening has no transcendental function, so FP64 is bit-identical to the oracle on every
cell and face.  FP32 bulk is held to the 1e-5 of the other FP32 tests over a few steps.
"""
import numpy as np
import pytest

import tmo
from tetemoko_amd import capi, scenarios

pytestmark = pytest.mark.gpu

G = scenarios.GHOST
NSTEPS = 4


def _case(nx, ny, boxes, bc, precision, plastic=False, march=None, cs=None):
    cfg = scenarios.config_c0(seed=3, nx=nx, ny=ny, dx=100.0)
    if cs is not None:
        cfg["cs"] = cs
    cfg["bc"] = bc
    if plastic:
        cfg.update(plasticity=1, p_mu=0.6, p_beta=0.3, p_eta=0.03 * scenarios.G_MPA, p_b=1.0)
    U, B = scenarios.level_arrays(cfg)
    scenarios.perturb(U, seed=nx * 1000 + ny, amp_v=1.0, amp_s=5.0)
    dt = scenarios.dt_of(cfg)
    Ur, Br = U.copy(), B.copy()
    assert tmo.level_steps(tmo.OracleParams(cfg), Ur, Br, 0.0, dt, NSTEPS) == 0
    ctx = capi.Context(cfg, precision)
    if march is not None:
        ctx.set_march(march)
    lev = capi.Level(ctx, boxes)
    for k, b in enumerate(boxes):
        lev.upload(k, scenarios.box_view(U, b), scenarios.box_bview(B, b) if b[1] == 0 else None)
    lev.run(NSTEPS, 0.0, dt)
    lev.sync()
    Ug, Bg = np.full_like(U, np.nan), np.full_like(B, np.nan)
    for k, (x0, y0, x1, y1) in enumerate(boxes):
        ub = scenarios.box_view(U, boxes[k])
        bb = scenarios.box_bview(B, boxes[k]) if y0 == 0 else None
        lev.download(k, ub, bb)
        Ug[:, y0 + G:y1 + G + 1, x0 + G:x1 + G + 1] = ub[:, G:-G, G:-G]
        if bb is not None:
            Bg[:, x0 + G:x1 + G + 1] = bb[:, G:-G]
    lev.close()
    ctx.close()
    s = (slice(None), slice(G, -G), slice(G, -G))
    return Ug[s], Ur[s], Bg[:, G:-G], Br[:, G:-G]


LAYOUTS = {
    "5x6": (5, 6, None),              # no cell's stencil lies inside the domain
    "7x7": (7, 7, None),              # one interior cell
    "24x8": (24, 8, None),            # a row band of 23 + 1 cells
    "23x29": (23, 29, None),          # row pieces of exactly 23, column pieces of 23
    "30x75": (30, 75, None),
    "65x31": (65, 31, None),          # a strip of 58 and one of 1
    "52x40 cut": (52, 40, [(0, 0, 23, 0), (24, 0, 51, 0), (0, 1, 51, 1), (0, 2, 22, 39), (23, 2, 51, 39)]),
    "52x40 boxes": (52, 40, scenarios.split_boxes(52, 40, 16)),
}


@pytest.mark.parametrize("bc", [(0, 0, 0, 0), (1, 0, 0, 1)])
@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_FP32_BULK])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_small_domains_and_cut_bands(layout, precision, bc):
    nx, ny, boxes = LAYOUTS[layout]
    Ug, Ur, Bg, Br = _case(nx, ny, boxes or [(0, 0, nx - 1, ny - 1)], bc, precision, plastic=nx > 50)
    if precision == capi.PREC_FP64:
        assert np.array_equal(Ug, Ur) and np.array_equal(Bg, Br)
        return
    scale = np.maximum(np.abs(Ur).reshape(22, -1).max(axis=1), 1e-300)
    err = np.abs(Ug - Ur).reshape(22, -1).max(axis=1) / scale
    assert np.all(err <= 1e-5), err


@pytest.mark.parametrize("nx,ny", [(64, 40), (300, 150), (1500, 700)])
def test_chosen_strip_height_changes_nothing(nx, ny):
    """The height a launch chooses by its size gives the state of a height set by hand (FP32 bulk:
    a cell's arithmetic does not depend on it)."""
    boxes = scenarios.split_boxes(nx, ny, 250)
    a = _case(nx, ny, boxes, (0, 0, 0, 0), capi.PREC_FP32_BULK)
    b = _case(nx, ny, boxes, (0, 0, 0, 0), capi.PREC_FP32_BULK, march=5)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("plastic", [False, True])
@pytest.mark.parametrize("cs", [scenarios.CS, 3013.5])
def test_divisions_of_either_kind(cs, plastic):
    """A shear speed whose impedance or density does not pass the check of the two-operation division
    (tests/test_div2.py), and the one every scenario has: both bit-identical to the oracle."""
    Ug, Ur, Bg, Br = _case(130, 70, [(0, 0, 129, 69)], (0, 0, 0, 0), capi.PREC_FP64, plastic=plastic, cs=cs)
    assert np.array_equal(Ug, Ur) and np.array_equal(Bg, Br)


@pytest.mark.parametrize("plastic", [False, True])
@pytest.mark.parametrize("nx,ny", [(64, 17), (65, 40), (121, 30), (122, 9)])
def test_fp32_march_no_further_off_than_the_tiles(nx, ny, plastic):
    """The FP32 march carries characteristics, the tile kernels (march=0) face states: at strips of 58
    columns and of one, the march is no further from the oracle than they are.  Both accumulate some 30
    roundings of 2^-24 a step that do not depend on one another, so the largest errors of the two differ
    by less than a factor of 2, up to one rounding a step."""
    boxes = [(0, 0, nx - 1, ny - 1)]
    errs = []
    for march in (6, 0):
        Ug, Ur, _, _ = _case(nx, ny, boxes, (0, 1, 0, 0), capi.PREC_FP32_BULK, plastic=plastic, march=march)
        scale = np.maximum(np.abs(Ur).reshape(22, -1).max(axis=1), 1e-300)
        errs.append(np.abs(Ug - Ur).reshape(22, -1).max(axis=1) / scale)
    assert np.all(errs[0] <= 2.0 * errs[1] + NSTEPS * 2.0 ** -24), errs


@pytest.mark.parametrize("fault", ["sw", "rs"])
@pytest.mark.parametrize("ghosts", [3, 4])
@pytest.mark.parametrize("valid", [(0, 0, 31, 31), (40, 0, 40, 0), (17, 0, 80, 70), (5, 3, 62, 20), (90, 60, 129, 79),
                                   (60, 1, 63, 79), (3, 3, 126, 76)])
def test_drop_in_call_marches_as_the_tiles(valid, ghosts, fault):
    """An FP64 drop-in call takes the marching step; set_march(0) keeps it on the tile kernels.  State,
    fluxes and slip-weakening fault data are the same bit for bit; boxes on edges and corners, of one
    cell, of more than 63 rows, inside; arrays of 4 ghosts and of the least a call accepts (3, cut off
    at the domain)."""
    nx, ny = 130, 80
    cfg = (scenarios.config_c0 if fault == "sw" else scenarios.config_c1)(seed=6, nx=nx, ny=ny, dx=50.0)
    U, B = scenarios.level_arrays(cfg)
    scenarios.perturb(U, seed=8, amp_v=1.0, amp_s=5.0)
    x0, y0, x1, y1 = valid
    ub = (x0 - ghosts, y0 - ghosts, x1 + ghosts, y1 + ghosts)
    if ghosts == 3:
        ub = (max(ub[0], 0), max(ub[1], 0), min(ub[2], nx - 1), min(ub[3], ny - 1))
    g = 1 if ghosts == 3 else G
    bb = (x0 - g, 0, x1 + g, 0)
    got = []
    for march in (None, 0):
        ctx = capi.Context(cfg, capi.PREC_FP64)
        if march is not None:
            ctx.set_march(march)
        Ub = np.ascontiguousarray(U[:, ub[1] + G:ub[3] + G + 1, ub[0] + G:ub[2] + G + 1])
        Bb = np.ascontiguousarray(B[:, bb[0] + G:bb[2] + G + 1]) if y0 == 0 else None
        F = [np.full((22, y1 - y0 + 1, x1 - x0 + 2), np.nan), np.full((22, y1 - y0 + 2, x1 - x0 + 1), np.nan)]
        ctx.update_state(valid, Ub, ub, Bb, bb if y0 == 0 else None, F[0], F[1], time=0.2, dt=scenarios.dt_of(cfg))
        ctx.close()
        got.append([Ub, Bb] + F)
    for k, (a, b) in enumerate(zip(*got)):
        if a is None:
            assert b is None
        elif fault == "sw" or y0 > 0:
            assert np.array_equal(a, b) and not np.isnan(a).any(), k
        else:  # the two builds of the rate-and-state solve: 1e-13 of the largest value, as against the oracle
            top = np.maximum(np.abs(b).reshape(b.shape[0], -1).max(axis=1), 1e-300)
            assert np.all(np.abs(a - b).reshape(b.shape[0], -1).max(axis=1) <= 1e-13 * top), k
