"""Reading a box back (tmk_level_download): its planes come in pieces of 1 MiB through pinned slots, by
one, two or four host threads, and FP32 levels add the background on the host.

The sizes: one piece; pieces that end inside a plane; two and four threads with a short last piece;
several boxes of one island; readers on several threads at once.  What is read is what was uploaded:
FP64 bit for bit, FP32 the background plus the difference rounded to FP32, both exact in NumPy.
"""
import threading

import numpy as np
import pytest

from tetemoko_amd import capi, scenarios

pytestmark = pytest.mark.gpu


def _check(nx, ny, precision, maxbox=0, seed=1):
    cfg = scenarios.config_c1(seed=seed, nx=nx, ny=ny, dx=25.0)
    U, B = scenarios.level_arrays(cfg)
    scenarios.perturb(U, seed=seed, amp_v=1.0, amp_s=5.0)
    boxes = scenarios.split_boxes(nx, ny, maxbox) if maxbox else [(0, 0, nx - 1, ny - 1)]
    ctx = capi.Context(cfg, precision)
    lev = capi.Level(ctx, boxes)
    for k, b in enumerate(boxes):
        lev.upload(k, scenarios.box_view(U, b), scenarios.box_bview(B, b) if b[1] == 0 else None)
    want = U
    if precision == capi.PREC_FP32_BULK:
        bg = scenarios.background_vector(cfg)[:, None, None]
        want = (U - bg).astype(np.float32).astype(np.float64) + bg
    ok = True
    for k, b in enumerate(boxes):
        Ub = np.full_like(scenarios.box_view(U, b), np.nan)
        Bb = np.full_like(scenarios.box_bview(B, b), np.nan) if b[1] == 0 else None
        lev.download(k, Ub, Bb)
        g = scenarios.GHOST
        ok = ok and np.array_equal(Ub[:, g:-g, g:-g], scenarios.box_view(want, b)[:, g:-g, g:-g])
        if Bb is not None:
            ok = ok and np.array_equal(Bb[:, g:-g], scenarios.box_bview(B, b)[:, g:-g])
    lev.close()
    ctx.close()
    return ok


@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_FP32_BULK])
@pytest.mark.parametrize("nx,ny,maxbox", [(9, 8, 0), (101, 73, 0), (257, 201, 0), (401, 333, 0), (300, 190, 97)])
def test_what_was_uploaded(nx, ny, maxbox, precision):
    assert _check(nx, ny, precision, maxbox)


def test_readers_on_several_threads():
    got = [None] * 6

    def run(t):
        got[t] = all(_check(150 + 40 * t, 90 + 31 * t, capi.PREC_FP64 if t % 2 else capi.PREC_FP32_BULK, seed=t + 1)
                     for _ in range(2))

    th = [threading.Thread(target=run, args=(t,)) for t in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert got == [True] * 6
    assert capi.lib().tmk_cache_trim() == 0
    assert _check(120, 80, capi.PREC_FP64)


@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_FP32_BULK])
@pytest.mark.parametrize("valid,flux", [((0, 0, 0, 0), True), ((5, 0, 37, 20), True), ((40, 17, 71, 50), False),
                                        ((3, 1, 95, 61), True)])
def test_drop_in_call_through_a_stage_and_by_copies(valid, flux, precision):
    """tmk_patch_update_state moves its data through a pinned stage; the allocation-free call copies when
    no stage is idle (tmk_cache_trim).  The same kernels on the same data: bit-identical, ghosts and
    untouched planes included."""
    g = scenarios.GHOST
    cfg = scenarios.config_c1(seed=9, nx=110, ny=70, dx=25.0)
    U, B = scenarios.level_arrays(cfg)
    scenarios.perturb(U, seed=4, amp_v=1.0, amp_s=5.0)
    x0, y0, x1, y1 = valid
    ub, bb = (x0 - g, y0 - g, x1 + g, y1 + g), (x0 - g, 0, x1 + g, 0)
    fault = y0 == 0
    ctx = capi.Context(cfg, precision)
    got = []
    for copies in (False, True):
        Ub = np.ascontiguousarray(U[:, y0:y1 + 2 * g + 1, x0:x1 + 2 * g + 1])
        Bb = np.ascontiguousarray(B[:, x0:x1 + 2 * g + 1]) if fault else None
        F = [np.full((22, y1 - y0 + 1, x1 - x0 + 2), np.nan), np.full((22, y1 - y0 + 2, x1 - x0 + 1), np.nan)]
        if copies:
            assert capi.lib().tmk_cache_trim() == 0
        ctx.update_state(valid, Ub, ub, Bb, bb if fault else None, *(F if flux else (None, None)), time=0.3,
                         dt=scenarios.dt_of(cfg), noalloc=copies)
        got.append([Ub, Bb] + (F if flux else []))
    ctx.close()
    for a, b in zip(*got):
        assert a is None and b is None or np.array_equal(a, b) and not np.isnan(a).any()


def test_more_readers_than_pinned_buffers():
    """24 readers at once on one device, which has 16 pinned buffers: those that find none copy through
    device memory (1 and 2 such pieces), with the same values."""
    n = 24
    got = [None] * n
    start = threading.Barrier(n)

    def run(t):
        precision = capi.PREC_FP64 if t % 2 else capi.PREC_FP32_BULK
        start.wait()
        got[t] = all(_check(90 + 11 * t, 70 + 7 * t, precision, seed=t + 1) for _ in range(3))

    th = [threading.Thread(target=run, args=(t,)) for t in range(n)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert got == [True] * n


@pytest.mark.parametrize("n", [40, 62, 66, 90])
def test_fp32_calls_on_both_sides_of_the_stage_limits(n):
    """FP32 calls without fault data and fluxes copy beyond 1 MiB of state, the plastic return beyond 5/8 MiB;
    the allocation-free call stages them: bit-identical, and so is a return through a stage and by copies."""
    g = scenarios.GHOST
    cfg = scenarios.config_c1(seed=9, nx=140, ny=120, dx=25.0)
    cfg.update(plasticity=1, p_mu=0.6, p_beta=0.3, p_eta=0.03 * scenarios.G_MPA, p_b=1.0)
    U, _ = scenarios.level_arrays(cfg)
    scenarios.perturb(U, seed=4, amp_v=1.0, amp_s=60.0)
    x0, y0, x1, y1 = 9, 8, 9 + n - 1, 8 + n - 1
    ub = (x0 - g, y0 - g, x1 + g, y1 + g)
    U0 = np.ascontiguousarray(U[:, y0:y1 + 2 * g + 1, x0:x1 + 2 * g + 1])
    dt = scenarios.dt_of(cfg)
    ctx = capi.Context(cfg, capi.PREC_FP32_BULK)
    a, b = U0.copy(), U0.copy()
    ctx.update_state((x0, y0, x1, y1), a, ub, time=0.3, dt=dt)
    ctx.update_state((x0, y0, x1, y1), b, ub, time=0.3, dt=dt, noalloc=True)
    assert np.array_equal(a, b) and not np.array_equal(a, U0)
    whole, parts = a.copy(), a.copy()
    ctx.plastic_update((x0, y0, x1, y1), whole, ub, dt)
    for y in range(y0, y1 + 1, 20):  # boxes small enough for a stage
        yt = min(y + 19, y1)
        sub = np.ascontiguousarray(parts[:, y - ub[1]:yt - ub[1] + 1])
        ctx.plastic_update((x0, y, x1, yt), sub, (ub[0], y, ub[2], yt), dt)
        parts[:, y - ub[1]:yt - ub[1] + 1] = sub
    ctx.close()
    s = (slice(None), slice(g, -g), slice(g, -g))
    assert np.array_equal(whole[s], parts[s]) and not np.array_equal(whole[s], a[s])
