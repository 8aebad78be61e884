"""Performance cases: the work a user of tetemoko_amd has it do, through its public entry points.

Kinds of case
  patch   the drop-in call on one box of host FArrayBox data (capi.Context.update_state, then
          plastic_update where the scenario has plasticity), one call per box and step as the
          reference's level loop makes it
  level   a device-resident level advanced by some steps (capi.Level.run), then read: the whole
          state and the fault data, or, for levels too large to read back at every interval,
          the fault data, the refinement tags and the station records
  amr     a three-level subcycled hierarchy (capi.Amr.run), read as the averaged-down base level
          and every level's fault data
  batch   several scenarios of the serving stream in shared launches (capi.Batch, or
          capi.AmrBatch for scenarios with refined levels): join, run, leave, fault data

Initial states of patches, levels and hierarchies are the configuration's background with a seeded
wave field everywhere, the state a running rupture is in (the largest levels' is set on the device,
one state per box, whose jumps send out the waves); batches start scenarios from the background
as the serving loop does.  Every pass goes on from where the last one ended.  Outputs of the reduced-precision mode
are given in float32, the precision its bulk carries.
"""
import math

import numpy as np
import torch

from tetemoko_amd import amr, amr_bench, capi, scenarios, serving

G = scenarios.GHOST


def listed():
    return [
        # drop-in call, one box of the reference's default size on the fault: latency of one call
        {"name": "patch_32x32_sw_fp64", "kind": "patch", "fault": "sw", "plastic": False, "precision": 64,
         "nx": 32, "ny": 32, "x0": 64, "flux": True, "noalloc": False},
        # drop-in call without device allocation, reduced precision, ragged box at the domain's corner
        {"name": "patch_93x61_rs_plastic_fp32", "kind": "patch", "fault": "rs", "plastic": True, "precision": 32,
         "nx": 93, "ny": 61, "x0": 0, "flux": False, "noalloc": True},
        # the slip-weakening configuration on one level, one plot interval
        {"name": "level_400x200_sw_fp64", "kind": "level", "fault": "sw", "plastic": False, "precision": 64,
         "nx": 400, "ny": 200, "steps": 300, "maxbox": 0, "read": "state", "stations": 0, "tune": False},
        # smallest grid of the serving stream, odd extents: many short steps
        {"name": "level_261x131_rs_fp32", "kind": "level", "fault": "rs", "plastic": False, "precision": 32,
         "nx": 261, "ny": 131, "steps": 400, "maxbox": 0, "read": "state", "stations": 0, "tune": False},
        # the base grid of the multi-level workload as one level of several boxes
        {"name": "level_1024x512_rs_plastic_fp32", "kind": "level", "fault": "rs", "plastic": True, "precision": 32,
         "nx": 1024, "ny": 512, "steps": 200, "maxbox": 256, "read": "state", "stations": 0, "tune": False},
        # ragged, full precision, no plasticity
        {"name": "level_1021x509_rs_fp64", "kind": "level", "fault": "rs", "plastic": False, "precision": 64,
         "nx": 1021, "ny": 509, "steps": 100, "maxbox": 0, "read": "state", "stations": 0, "tune": False},
        # the plain full-precision drop-in configuration between two regrids, with stations
        {"name": "level_4096x2048_rs_fp64", "kind": "level", "fault": "rs", "plastic": False, "precision": 64,
         "nx": 4096, "ny": 2048, "steps": 60, "maxbox": 128, "read": "tags", "stations": 48, "tune": False},
        # the benchmark's workload in both precisions, tuned as the benchmark tunes it
        {"name": "level_8192x4096_rs_plastic_fp64", "kind": "level", "fault": "rs", "plastic": True, "precision": 64,
         "nx": 8192, "ny": 4096, "steps": 50, "maxbox": 128, "read": "tags", "stations": 0, "tune": True},
        {"name": "level_8192x4096_rs_plastic_fp32", "kind": "level", "fault": "rs", "plastic": True, "precision": 32,
         "nx": 8192, "ny": 4096, "steps": 100, "maxbox": 128, "read": "fault", "stations": 0, "tune": True},
        # the multi-level workload: three levels, ratio 4, several hundred uneven boxes
        {"name": "amr_1024x512_r4_rs_plastic_fp32", "kind": "amr", "fault": "rs", "plastic": True, "precision": 32,
         "nx": 1024, "ny": 512, "ratio": 4, "steps": 12},
        # serving: a wave of single-level scenarios of mixed sizes and friction laws
        {"name": "batch_12_single_fp32", "kind": "batch", "precision": 32, "members": 12, "levels": 0, "steps": 200,
         "most": 2048, "mix": 1},
        # serving: a wave of scenarios with two refined levels each
        {"name": "batch_8_refined_fp32", "kind": "batch", "precision": 32, "members": 8, "levels": 2, "steps": 20,
         "most": 1024, "mix": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["patch", "level", "level", "level", "level", "amr", "batch"])
    precision = rng.choice([32, 64])
    if kind == "patch":
        return {"kind": "patch", "fault": rng.choice(["rs", "sw"]), "plastic": rng.random() < 0.5,
                "precision": precision, "nx": _log_int(rng, 8, 128), "ny": _log_int(rng, 8, 96),
                "x0": rng.choice([0, rng.randrange(1, 120)]), "flux": rng.random() < 0.5, "noalloc": rng.random() < 0.5}
    if kind == "level":
        nx = _log_int(rng, 200, 4096)
        ny = max(64, int(nx * rng.uniform(0.3, 0.7)))
        cells = nx * ny
        # about 1e8 cell-steps a pass where that is between 20 and 400 steps
        steps = max(20, min(400, int(1e8 / cells) + rng.randrange(0, 7)))
        fault = rng.choice(["rs", "rs", "sw"])
        return {"kind": "level", "fault": fault, "plastic": rng.random() < 0.5,
                "precision": precision, "nx": nx, "ny": ny, "steps": steps,
                "maxbox": rng.choice([0, 256, 257] if cells <= SMALL else [128, 192]),
                "read": "state" if cells <= SMALL else ("tags" if precision == 64 else "fault"),
                "stations": rng.choice([0, 48]), "tune": False}
    if kind == "amr":
        return {"kind": "amr", "fault": rng.choice(["rs", "sw"]), "plastic": rng.random() < 0.5,
                "precision": precision, "nx": rng.choice([256, 384, 512, 768]), "ny": rng.choice([192, 256, 384]),
                "ratio": rng.choice([2, 4]), "steps": rng.randrange(6, 13)}
    levels = rng.choice([0, 1, 2])
    return {"kind": "batch", "precision": precision, "members": rng.randrange(3, 11), "levels": levels,
            "steps": rng.randrange(50, 200) if levels == 0 else rng.randrange(8, 20), "most": rng.choice([512, 768, 1024]),
            "mix": rng.randrange(3, 1000)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _precision(case):
    return capi.PREC_FP64 if case["precision"] == 64 else capi.PREC_FP32_BULK


def _config(case, seed, nx, ny):
    """The repository's scenario of this friction law, grid and rheology, its per-face values seeded."""
    seed %= 1 << 20
    if case["fault"] == "sw":
        cfg = scenarios.config_c0(seed, nx, ny, 100.0)
    else:
        cfg = scenarios.config_c1(seed, nx, ny, 25.0)
    if case["plastic"]:
        cfg.update(plasticity=1, p_mu=0.6, p_beta=0.3, p_eta=0.03 * cfg["G"], p_b=1.0)
    return cfg


WAVES = 3  # of each component


def _field(seed, cfg, x, y, noise=0.0):
    """(22, len(y), len(x)) states at the base grid's cell coordinates x, y: the background with waves
    of 16 to 200 cells on top, velocities of up to 0.02 m/s and stresses of up to 0.2 MPa (in
    proportion through the impedance), and white noise of that share of them."""
    rng = np.random.default_rng([seed, 5])
    u = np.empty((22, len(y), len(x)))
    u[:] = scenarios.background_vector(cfg)[:, None, None]
    for s in (0, 11):
        for c, a in ((0, 0.02), (1, 0.02), (3, 0.2), (4, 0.2), (5, 0.2), (6, 0.2)):
            for _ in range(WAVES):
                k, l = 2.0 * math.pi / np.exp(rng.uniform(math.log(16.0), math.log(200.0), 2))
                p, q = rng.uniform(0.0, 6.28, 2)
                u[s + c] += np.outer(np.sin(l * y + q), (a / WAVES) * np.sin(k * x + p))
            if noise:
                u[s + c] += rng.uniform(-noise * a, noise * a, u.shape[1:])
    return u


SMALL = 1 << 20  # cells up to which a level's initial state comes from the host


def _initial(case, seed, cfg):
    """A level's initial state, (22, ny, nx) without ghosts.  Larger levels, whose state is set on the
    device, hold one seeded state per box: _box_states."""
    return _field(seed, cfg, np.arange(case["nx"]), np.arange(case["ny"]), 0.05)


def _box_states(seed, cfg, n):
    rng = np.random.default_rng([seed, 5])
    u = np.broadcast_to(scenarios.background_vector(cfg), (n, 22)).copy()
    for s in (0, 11):
        u[:, s:s + 2] += rng.uniform(-0.02, 0.02, (n, 2))
        u[:, s + 3:s + 7] += rng.uniform(-0.2, 0.2, (n, 4))
    return u


def _patch_inputs(case, seed):
    """Host arrays of one box (ghosted by 4) of a level four times its size, on the fault."""
    nx, ny, x0 = case["nx"], case["ny"], case["x0"]
    cfg = _config(case, seed, x0 + 2 * nx + 16, 2 * ny + 16)
    rng = np.random.default_rng([seed, 7])
    U = np.empty((22, ny + 2 * G, nx + 2 * G))
    U[:] = scenarios.background_vector(cfg)[:, None, None]
    y = np.linspace(0.0, 1.0, U.shape[1])[:, None]
    x = np.linspace(0.0, 1.0, U.shape[2])[None, :]
    for s in (0, 11):
        for c, a in ((0, 0.05), (1, 0.05), (3, 0.5), (4, 0.5), (5, 0.5), (6, 0.5)):
            k, l, p = rng.uniform(2.0, 40.0), rng.uniform(2.0, 40.0), rng.uniform(0.0, 6.28)
            U[s + c] += a * np.sin(k * x + l * y + p) + rng.uniform(-0.05 * a, 0.05 * a, U.shape[1:])
    B = np.ascontiguousarray(scenarios.fault_arrays(cfg)[:, x0:x0 + nx + 2 * G])
    return cfg, U, B


def _scenarios(case, seed):
    """(scenario, box layout) of a batch's members: grids, friction laws and nucleations as the serving
    stream draws them (the case's mix), per-face values from the seed."""
    out = []
    for sc in serving.draw_scenarios(case["members"], case["mix"], nx_range=(256, case["most"]), max_levels=0):
        sc["levels"] = case["levels"]
        cfg, k = sc["cfg"], (seed % (1 << 16)) * 100 + sc["id"]
        nx, ny, dx = cfg["nx"], cfg["ny"], cfg["dx"]
        if cfg["fault"] == "sw":
            new = scenarios.config_c0(k, nx, ny, dx)
            new["faces"]["tau"] = np.roll(new["faces"]["tau"], sc["xn"] - nx // 2)
        else:
            new = scenarios.config_c1(k, nx, ny, dx)
            new["rs"].update(nuc_x=cfg["rs"]["nuc_x"], nuc_R=cfg["rs"]["nuc_R"])
        sc["cfg"] = new
        out.append((sc, serving.amr_layout(sc)))
    return out


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    kind = case["kind"]
    if kind == "patch":
        cfg, s.U0, s.B0 = _patch_inputs(case, seed)
        s.ctx = capi.Context(cfg, _precision(case))
        nx, ny, x0 = case["nx"], case["ny"], case["x0"]
        s.box = (x0, 0, x0 + nx - 1, ny - 1)
        s.ubox = (x0 - G, -G, x0 + nx - 1 + G, ny - 1 + G)
        s.bbox = (x0 - G, 0, x0 + nx - 1 + G, 0)
        s.dt = scenarios.dt_of(cfg)
        s.U, s.B = s.U0.copy(), s.B0.copy()
        s.F = (np.zeros((22, ny, nx + 1)), np.zeros((22, ny + 1, nx))) if case["flux"] else (None, None)
        return s
    if kind == "level":
        nx, ny = case["nx"], case["ny"]
        cfg = _config(case, seed, nx, ny)
        s.ctx = capi.Context(cfg, _precision(case))
        boxes = scenarios.split_boxes(nx, ny, case["maxbox"]) if case["maxbox"] else [(0, 0, nx - 1, ny - 1)]
        s.lev = capi.Level(s.ctx, boxes)
        B = scenarios.fault_arrays(cfg)
        large = nx * ny > SMALL
        if large:
            w = _box_states(seed, cfg, len(boxes))
        else:
            U = np.empty((22, ny + 2 * G, nx + 2 * G))
            U[:] = scenarios.background_vector(cfg)[:, None, None]
            U[:, G:-G, G:-G] = _initial(case, seed, cfg)
        for k, b in enumerate(boxes):
            bb = scenarios.box_bview(B, b) if b[1] == 0 else None
            if large:
                s.lev.fill(k, w[k], bb)
            else:
                s.lev.upload(k, scenarios.box_view(U, b), bb)
        s.dt, s.t = scenarios.dt_of(cfg), 0.0
        if case["tune"]:
            s.lev.autotune(0.0, s.dt)
        nb = scenarios.NB[cfg["fault"]]
        s.boxes = boxes
        s.fault = [(k, np.empty((nb, b[2] - b[0] + 1 + 2 * G))) for k, b in enumerate(boxes) if b[1] == 0]
        s.state = None
        if case["read"] == "state":
            s.state = [np.empty((22, b[3] - b[1] + 1 + 2 * G, b[2] - b[0] + 1 + 2 * G)) for b in boxes]
        s.stations = None
        if case["stations"]:
            x = np.sort(np.random.default_rng([seed, 9]).uniform(2.0, nx - 2.0, case["stations"])) * cfg["dx"]
            s.stations = capi.Stations(s.lev, x, case["steps"])
        if case["read"] == "tags":
            s.tag = capi.TagParams.make(refine_thresh=0.01, tag_buffer=2, sliprate_thresh=1e-3)
        return s
    if kind == "amr":
        nx, ny, r = case["nx"], case["ny"], case["ratio"]
        cfg = _config(case, seed, nx, ny)
        dx, xc = cfg["dx"], 0.5 * nx * cfg["dx"]
        w = nx * dx / 25600.0  # the multi-level workload's lenses, in proportion to the grid
        boxes = [scenarios.split_boxes(nx, ny, 64)]
        for l, (half, hc, he) in enumerate(((9600.0, 2000.0, 500.0), (6400.0, 800.0, 200.0)), 1):
            m = amr_bench.lens_mask(nx * r ** l, ny * r ** l, dx / r ** l, xc, half * w, hc * w, he * w)
            boxes.append(amr_bench.tile_boxes(m))
        s.ctxs, s.levels = amr.make_levels(cfg, boxes, r, _precision(case))
        s.fault = []
        lcfg = cfg
        for l, lev in enumerate(s.levels):
            lcfg = cfg if l == 0 else scenarios.refine_cfg(lcfg, r)
            B = scenarios.fault_arrays(lcfg)
            f = 1.0 / r ** l
            for k, b in enumerate(boxes[l]):
                bb = scenarios.box_bview(B, b) if b[1] == 0 else None
                x = (np.arange(b[0] - G, b[2] + G + 1) + 0.5) * f - 0.5
                y = (np.arange(b[1] - G, b[3] + G + 1) + 0.5) * f - 0.5
                lev.upload(k, _field(seed, cfg, x, y), bb)
                if bb is not None:
                    s.fault.append((l, k, bb))
        s.amr = capi.Amr(s.levels, r)
        s.boxes = boxes[0]
        s.state = [np.empty((22, b[3] - b[1] + 1 + 2 * G, b[2] - b[0] + 1 + 2 * G)) for b in s.boxes]
        s.dt, s.t = scenarios.dt_of(cfg), 0.0
        return s
    s.members = []
    for sc, layout in _scenarios(case, seed):
        ctxs, levels = amr.make_levels(sc["cfg"], layout, serving.AMR_RATIO, _precision(case))
        nb = scenarios.NB[sc["cfg"]["fault"]]
        fault = [(l, k, np.empty((nb, b[2] - b[0] + 1 + 2 * G)))
                 for l, bl in enumerate(layout) for k, b in enumerate(bl) if b[1] == 0]
        s.members.append((ctxs, levels, scenarios.dt_of(sc["cfg"]), fault))
    s.batch = capi.Batch() if case["levels"] == 0 else capi.AmrBatch(case["levels"] + 1, serving.AMR_RATIO)
    s.t = [0.0] * len(s.members)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _out(case, a):
    return a if case["precision"] == 64 else a.astype(np.float32)


def _clock(t, dt, steps):
    """The time the framework's own clocks reach: one addition a step (another time would restart a
    hierarchy)."""
    for _ in range(steps):
        t = t + dt
    return t


def _fields(case, u):
    """A state array's planes by what they hold (views): velocities and the rest, per side."""
    return {"velocity1": _out(case, u[0:3]), "stress1": _out(case, u[3:11]),
            "velocity2": _out(case, u[11:14]), "stress2": _out(case, u[14:22])}


def _box_fields(case, u):
    """The same of one of several boxes, in two parts."""
    return {"velocity1": _out(case, u[0:3]), "rest": _out(case, u[3:22])}


def _fault(case, parts):
    """The fault faces of several boxes side by side, without their ghosts: the rupture times apart
    (a face that has not ruptured holds 1e10)."""
    b = np.concatenate([p[:, G:-G] for p in parts], axis=1)
    return _fault_fields(case, b)


def _fault_fields(case, b):
    t = 9 if b.shape[0] == scenarios.NB["rs"] else 8
    return {"rows": _out(case, b[:t]), "time": _out(case, b[t]), "state": _out(case, b[t + 1:])}


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "patch":
        np.copyto(s.U, s.U0)  # the level's data of this step
        np.copyto(s.B, s.B0)
        s.ctx.update_state(s.box, s.U, s.ubox, s.B, s.bbox, s.F[0], s.F[1], 0.0, s.dt, noalloc=case["noalloc"])
        if case["plastic"]:
            s.ctx.plastic_update(s.box, s.U, s.ubox, s.dt)
        out = {"state": _fields(case, s.U[:, G:-G, G:-G]), "fault": _fault(case, [s.B])}
        if case["flux"]:
            out["flux_x"], out["flux_y"] = _out(case, s.F[0]), _out(case, s.F[1])
        return out
    if kind == "level":
        s.lev.run(case["steps"], s.t, s.dt)
        s.lev.sync()
        s.t = _clock(s.t, s.dt, case["steps"])
        out = {}
        if case["read"] == "state":
            faults = dict(s.fault)
            for k, u in enumerate(s.state):
                s.lev.download(k, u, faults.get(k))
            if not case["maxbox"]:
                out["state"] = _fields(case, s.state[0][:, G:-G, G:-G])
            else:
                out["state"] = [_box_fields(case, u[:, G:-G, G:-G]) for u in s.state]
        else:
            for k, b in s.fault:
                s.lev.download_fault(k, b)
        out["fault"] = _fault(case, [b for _, b in s.fault])
        if case["read"] == "tags":
            out["tags"] = s.lev.tag(s.tag, case["nx"], case["ny"])
        if s.stations is not None:
            out["records"] = _out(case, s.stations.read())
        return out
    if kind == "amr":
        s.amr.run(case["steps"], s.t, s.dt)
        s.amr.sync()
        s.t = _clock(s.t, s.dt, case["steps"])
        for k, u in enumerate(s.state):
            s.levels[0].download(k, u)
        for l, k, b in s.fault:
            s.levels[l].download_fault(k, b)
        out = {"state": _fields(case, _grid(case, s.boxes, s.state))}
        for l in range(len(s.levels)):
            out["fault%d" % l] = _fault(case, [b for m, _, b in s.fault if m == l])
        return out
    for m, (ctxs, levels, dt, fault) in enumerate(s.members):
        if case["levels"] == 0:
            s.batch.add(levels[0], s.t[m], dt)
        else:
            s.batch.add(levels, s.t[m], dt)
    if case["levels"] == 0:
        s.batch.run(case["steps"])
    else:
        s.batch.advance(case["steps"])
    s.batch.sync()
    out = []
    for m, (ctxs, levels, dt, fault) in enumerate(s.members):
        s.batch.remove(levels[0])
        s.t[m] = _clock(s.t[m], dt, case["steps"])
        for l, k, b in fault:
            levels[l].download_fault(k, b)
        out.append(_fault(case, [b for _, _, b in fault]))
    return out


def _grid(case, boxes, parts):
    out = np.empty((22, case["ny"], case["nx"]))
    for (x0, y0, x1, y1), u in zip(boxes, parts):
        out[:, y0:y1 + 1, x0:x1 + 1] = u[:, G:-G, G:-G]
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# operations of one cell (both sides) and step: slopes, face values and limiting of four fields in
# two directions, tracing, four Riemann states, the transverse terms, the flux difference; the return
STEP_FLOPS, PLASTIC_FLOPS = 2 * 300, 2 * 50


def _cell(plastic, precision):
    """Bytes (the planes a step reads and writes, each once: 12 without plasticity, 15 with) and
    operations of one cell's step."""
    planes = 30 if plastic else 24
    return planes * precision // 8, STEP_FLOPS + (PLASTIC_FLOPS if plastic else 0)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        cells = 0
        for _, layout in _scenarios(case, 0):
            for l, bl in enumerate(layout):
                cells += sum((b[2] - b[0] + 1) * (b[3] - b[1] + 1) for b in bl) * serving.AMR_RATIO ** l
        b, f = _cell(False, case["precision"])
        return {"bytes": cells * b * case["steps"], "flops": cells * f * case["steps"]}
    b, f = _cell(case["plastic"], case["precision"])
    if kind == "patch":
        n = case["nx"] * case["ny"]
        ghosted = (case["nx"] + 2 * G) * (case["ny"] + 2 * G)
        return {"bytes": 22 * 8 * (n + ghosted) + (2 * 22 * 8 * n if case["flux"] else 0), "flops": n * f}
    if kind == "level":
        n = case["nx"] * case["ny"]
        read = 22 * 8 * n if case["read"] == "state" else n if case["read"] == "tags" else 0
        return {"bytes": n * b * case["steps"] + read, "flops": n * f * case["steps"]}
    nx, ny, r = case["nx"], case["ny"], case["ratio"]
    # the lenses' areas: half length x mean height on each side of the nucleation
    unit = (nx / 1024.0) ** 2 / 625.0
    areas = [nx * ny, min(2 * 9600.0 * 1250.0 * unit, nx * ny) * r ** 2, min(2 * 6400.0 * 500.0 * unit, nx * ny) * r ** 4]
    cells = sum(a * r ** l for l, a in enumerate(areas))
    return {"bytes": cells * b * case["steps"] + 22 * 8 * nx * ny, "flops": cells * f * case["steps"]}


# ---------------------------------------------------------------------------
# the same step in plain torch, 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "patch":
        cfg, U, B = _patch_inputs(case, seed)
        gx, gy = (0 if case["x0"] else G), G  # cells outside the domain are not part of the step
        if case["x0"] and case["x0"] < G:
            gx = G - case["x0"]
        e = _Exact(cfg, U[:, gy:, gx:], B[:, gx:], case["x0"] - G + gx)
        e.step(0.0, scenarios.dt_of(cfg), plastic=False)
        if case["plastic"]:
            # the return acts on the box's own cells
            e.plastic(scenarios.dt_of(cfg))
        nx, ny, o = case["nx"], case["ny"], G - gx
        wide = dict(case, precision=64)
        out = {"state": _fields(wide, e.state()[:, :ny, o:o + nx]), "fault": _fault_fields(wide, e.B[:, o:o + nx])}
        if case["flux"]:
            out["flux_x"] = e.flux(0)[:, :ny, o:o + nx + 1]
            out["flux_y"] = e.flux(1)[:, :ny + 1, o:o + nx]
        return out
    if case["kind"] != "level":
        return None
    nx, ny = case["nx"], case["ny"]
    cfg = _config(case, seed, nx, ny)
    if nx * ny > SMALL:
        return None
    e = _Exact(cfg, _initial(case, seed, cfg), scenarios.fault_arrays(cfg)[:, G:-G], 0)
    dt = scenarios.dt_of(cfg)
    t = 0.0
    for _ in range(case["steps"]):
        e.step(t, dt, plastic=case["plastic"])
        t = t + dt
    wide = dict(case, precision=64)
    out = {"fault": _fault_fields(wide, e.B)}
    if case["read"] == "state":
        u = e.state()
        if case["maxbox"]:
            out["state"] = [_box_fields(wide, u[:, b[1]:b[3] + 1, b[0]:b[2] + 1])
                            for b in scenarios.split_boxes(nx, ny, case["maxbox"])]
        else:
            out["state"] = _fields(wide, u)
    return out


class _Exact:
    """The Godunov step of a whole grid (mode II, PPM with primitive limiting, absorbing edges, the
    fault along the lower one) on (ny, nx) torch arrays in 64 bits."""

    def __init__(self, cfg, U, B, x0):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(np.array(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.cfg = cfg
        self.bg = scenarios.background_vector(cfg)
        self.u = [dict(zip(("vx", "vy", "sxx", "syy", "szz", "sxy", "lam", "gam"),
                           (t(U[11 * s + c]) for c in (0, 1, 3, 4, 5, 6, 9, 10)))) for s in (0, 1)]
        self.B = t(B)
        self.i = torch.arange(x0, x0 + U.shape[2], device=dev)
        cs, cp, self.G = cfg["cs"], cfg["cp"], cfg["G"]
        self.rho = self.G / cs ** 2
        self.lame = self.rho * cp ** 2 - 2 * self.G
        self.c = (cp, cs)
        self.Z = (self.rho * cp, self.rho * cs)
        self.face = {k: t(v)[torch.clamp(self.i - int(cfg["faces"]["lo"]), 0, len(v) - 1)]
                     for k, v in cfg.get("faces", {}).items() if k != "lo"}

    # shift along dimension d (0: x, 1: y): element i - 1 / i + 1, the edge's own at the edge
    @staticmethod
    def _prev(a, d):
        return torch.cat((a[:, :1], a[:, :-1]), 1) if d == 0 else torch.cat((a[:1], a[:-1]), 0)

    @staticmethod
    def _next(a, d):
        return torch.cat((a[:, 1:], a[:, -1:]), 1) if d == 0 else torch.cat((a[1:], a[-1:]), 0)

    def _ppm(self, w, d):
        """Limited increments of the lo and hi face values of every cell."""
        ax = 1 - d
        lo, hi = self._prev(w, d), self._next(w, d)
        l, r = w - lo, hi - w
        n = w.shape[ax]
        first, last = (slice(None), slice(0, 1)), (slice(None), slice(n - 1, n))
        if d == 1:
            first, last = first[::-1], last[::-1]
        s = torch.where(l * r > 0, torch.sign(l) * torch.minimum(2 * torch.minimum(l.abs(), r.abs()),
                                                                 (0.5 * (l + r)).abs()), torch.zeros_like(l))
        s[first], s[last] = r[first], l[last]
        fl = 0.5 * (w + lo) + (self._prev(s, d) - s) / 6
        fh = 0.5 * (hi + w) + (s - self._next(s, d)) / 6
        fl[first] = w[first] - 0.5 * s[first]
        fh[last] = w[last] + 0.5 * s[last]
        m, p = fl - w, fh - w
        keep = m * p < 0
        zero = torch.zeros_like(m)
        return (torch.where(keep, torch.sign(m) * torch.minimum(2 * p.abs(), m.abs()), zero),
                torch.where(keep, torch.sign(p) * torch.minimum(2 * m.abs(), p.abs()), zero))

    def _fields(self, side, d):
        """The two pairs (velocity, traction) of direction d."""
        u = self.u[side]
        return ((u["vx"], u["sxx"]), (u["vy"], u["sxy"])) if d == 0 else ((u["vy"], u["syy"]), (u["vx"], u["sxy"]))

    def _predict(self, side, d, r, dtdx):
        """W- and W+ of every cell: [pair][lo/hi] of (v, s)."""
        out = []
        for k, (v, s) in enumerate(self._fields(side, d)):
            vm, vp = self._ppm(v, d)
            sm, sp = self._ppm(s, d)
            rz = r * self.Z[k]
            am, bm, ap, bp = sm + rz * vm, sm - rz * vm, sp + rz * vp, sp - rz * vp
            g = self.c[k] * dtdx
            tm = am + 0.5 * g * ((ap - am) - (ap + am) * (3 - 2 * g))
            tp = bp + 0.5 * g * ((bm - bp) - (bp + bm) * (3 - 2 * g))
            out.append([[v + (tm - bm) / (2 * rz), s + 0.5 * (tm + bm)], [v + (ap - tp) / (2 * rz), s + 0.5 * (ap + tp)]])
        return out

    def _faces(self, W, side, d, r, fault=None):
        """Face states [pair] of (v, s) on all faces; fault(states of the lower row) gives the lo-y ones."""
        out = []
        for k in range(2):
            rz = r * self.Z[k]
            (vm, sm), (vp, sp) = W[k]
            right, left = sp - rz * vp, sm + rz * vm
            comp = ((0, 3), (1, 6)) if d == 0 else ((1, 4), (0, 6))
            bv, bs = (float(self.bg[11 * side + c]) for c in comp[k])
            cat = lambda a, b: torch.cat((a, b), 1 - d)  # noqa: E731
            edge = (lambda a: a[:, :1]) if d == 0 else (lambda a: a[:1])
            wp = cat(torch.full_like(edge(right), bs - rz * bv), right)
            wm = cat(left, torch.full_like(edge(left), bs + rz * bv))
            out.append([(wm - wp) / (2 * rz), 0.5 * (wm + wp)])
        if fault is not None:
            for k in range(2):
                out[k][0][0], out[k][1][0] = fault[k]
        return out

    def _transverse(self, W, H, d2, sc):
        """The predictor of the other direction corrected with the face states of direction d2."""
        df = (lambda a: a[:, 1:] - a[:, :-1]) if d2 == 0 else (lambda a: a[1:] - a[:-1])
        dn, ds = [df(a) for a in H[0]], [df(a) for a in H[1]]
        out = []
        for k, (dv, dsg) in enumerate(((sc * ds[1] / self.rho, sc * self.lame * dn[0]),
                                       (sc * dn[1] / self.rho, sc * self.G * ds[0]))):
            out.append([[v - dv, s - dsg] for v, s in W[k]])
        return out

    def _x(self):
        return (self.i.double() + 0.5) * self.cfg["dx"]

    def _fault(self, W, state):
        """Fault states per side and pair from the lower row's W- of both sides, the slip rate and
        the tractions."""
        Zp, Zs = self.Z
        vy, syy = zip(*((w[0][0][0][0], w[0][0][1][0]) for w in W))
        vx, sxy = zip(*((w[1][0][0][0], w[1][0][1][0]) for w in W))
        px1, py1 = -sxy[0] - Zs * vx[0], -syy[0] - Zp * vy[0]
        px2, py2 = sxy[1] - Zs * vx[1], syy[1] - Zp * vy[1]
        n, w = -(py1 - py2) / 2, -(py1 + py2) / (2 * Zp)
        bulk = 0.5 * (px2 - px1)
        tau0 = self.tau0()
        sn = -(n + self.face.get("syy", 0.0))
        if self.cfg["fault"] == "rs":
            phi = (bulk + tau0).abs()
            a = self.face["a"]
            V = self._newton(phi, state, sn, a, (vx[0] - vx[1]).abs())
            tau = sn * a * torch.asinh(torch.exp(state / a) / (2 * self.cfg["rs"]["V0"]) * V)
            sgn = (bulk + tau0) / phi
            s = sgn * tau - tau0
            x1 = -(s + px1) / Zs
            x2 = x1 - sgn * V
        else:
            f = self.face["fs"]
            f = f - (f - self.face["fd"]) * torch.clamp(state / self.face["dc"], max=1.0)
            tau = torch.minimum((bulk + tau0).abs(), sn * f) - tau0
            s = bulk / bulk.abs() * tau
            x1, x2 = -(s + px1) / Zs, (s - px2) / Zs
        return ([(w, n), (x1, s)], [(w, n), (x2, s)]), x1 - x2

    def tau0(self):
        t = self.face.get("tau", torch.zeros_like(self.B[0]))
        if self.cfg["fault"] == "rs":
            rs = self.cfg["rs"]
            t = t + rs["nuc_S"] * torch.exp(-0.5 * ((self._x() - rs["nuc_x"]) / rs["nuc_R"]) ** 2)
        return t

    def _newton(self, phi, psi, sn, a, V):
        """The root of sn a asinh(beta V) + Zs V / 2 = phi in [0, phi / Zs], safeguarded."""
        lo, hi = torch.zeros_like(phi), phi / self.Z[1]
        beta, eta = torch.exp(psi / a) / (2 * self.cfg["rs"]["V0"]), 0.5 * self.Z[1]
        V = torch.where((V < lo) | (V > hi), 0.5 * (lo + hi), V)
        for _ in range(100):
            f = sn * a * torch.asinh(beta * V) + eta * V - phi
            lo, hi = torch.where(f < 0, V, lo), torch.where(f < 0, hi, V)
            N = V - f / (sn * a * beta / torch.sqrt(beta * beta * V * V + 1) + eta)
            N = torch.where((N < lo) | (N > hi), 0.5 * (lo + hi), N)
            if torch.equal(N, V):
                break
            V = N
        return V

    def _psi(self, psi, V, dt):
        rs = self.cfg["rs"]
        return psi + dt * self.face["b"] * rs["V0"] / self.face["L"] * (torch.exp((rs["f0"] - psi) / self.face["b"]) - V / rs["V0"])

    def step(self, time, dt, plastic):
        cfg = self.cfg
        dtdx = dt / cfg["dx"]
        sgn = (1.0, -1.0)
        rs = cfg["fault"] == "rs"
        state = self.B[10] if rs else self.B[7]
        X = [self._predict(s, 0, 1.0, dtdx) for s in (0, 1)]
        Y = [self._predict(s, 1, sgn[s], dtdx) for s in (0, 1)]
        f, Vx = self._fault(Y, state)
        half = self._psi(state, Vx.abs(), 0.5 * dt) if rs else state + 0.5 * dt * Vx.abs()
        H0 = [self._faces(X[s], s, 0, 1.0) for s in (0, 1)]
        H1 = [self._faces(Y[s], s, 1, sgn[s], f[s]) for s in (0, 1)]
        X = [self._transverse(X[s], H1[s], 1, -0.5 * dtdx * sgn[s]) for s in (0, 1)]
        Y = [self._transverse(Y[s], H0[s], 0, -0.5 * dtdx) for s in (0, 1)]
        f, Vx = self._fault(Y, half)
        self.F = [[self._faces(X[s], s, 0, 1.0) for s in (0, 1)],
                  [self._faces(Y[s], s, 1, sgn[s], f[s]) for s in (0, 1)]]
        self._set_fault(time, dt, f, Vx)
        k = dtdx
        for s in (0, 1):
            (xn, xns), (xs, xss) = [[a[:, 1:] - a[:, :-1] for a in p] for p in self.F[0][s]]
            (yn, yns), (ys, yss) = [[sgn[s] * (a[1:] - a[:-1]) for a in p] for p in self.F[1][s]]
            u = self.u[s]
            l2 = self.lame + 2 * self.G
            u["vx"] = u["vx"] + k / self.rho * (xns + yss)
            u["vy"] = u["vy"] + k / self.rho * (xss + yns)
            u["sxx"] = u["sxx"] + k * (l2 * xn + self.lame * yn)
            u["syy"] = u["syy"] + k * (self.lame * xn + l2 * yn)
            u["szz"] = u["szz"] + k * self.lame * (xn + yn)
            u["sxy"] = u["sxy"] + k * self.G * (xs + ys)
        if plastic:
            self.plastic(dt)

    def _set_fault(self, time, dt, f, Vx):
        V, new, B = Vx.abs(), time + dt, self.B.clone()
        zero = torch.zeros_like(V)
        n, s = f[0][0][1], f[0][1][1]
        if self.cfg["fault"] == "rs":
            rows = [Vx, zero, V, s + self.tau0(), zero, n, B[6] + dt * Vx, B[7], B[8] + dt * V,
                    torch.where((B[9] > new) & (V > self.cfg["rs"]["rupture_thr"]), new,
                                torch.where(B[9] > new, 1e10, B[9])), self._psi(B[10], V, dt)]
        else:
            rows = [Vx, zero, s, zero, V, B[5] + dt * Vx, B[6], B[7] + dt * V,
                    torch.where((B[8] > new) & (V > self.cfg["sw"]["rupture_thr"]), new, B[8])]
        self.B = torch.stack(rows)

    def plastic(self, dt):
        c = self.cfg
        K = self.lame + 2 * self.G / 3
        for u in self.u:
            m = (u["sxx"] + u["syy"] + u["szz"]) / 3
            dev = {k: u[k] - m for k in ("sxx", "syy", "szz")}
            J2 = ((u["sxx"] - u["syy"]) ** 2 + (u["syy"] - u["szz"]) ** 2 + (u["szz"] - u["sxx"]) ** 2) / 6 + u["sxy"] ** 2
            tau = torch.sqrt(J2)
            Y = tau - torch.clamp(-c["p_mu"] * m + c["p_b"], min=0.0)
            lam = torch.where(Y > 0, Y / (dt * (self.G + c["p_mu"] * c["p_beta"] * K) + c["p_eta"]), torch.zeros_like(Y))
            u["lam"], u["gam"] = lam, u["gam"] + dt * lam
            f = torch.where(Y > 0, (tau - dt * lam * self.G) / tau, torch.ones_like(tau))
            for k in dev:
                u[k] = m - dt * lam * K * c["p_beta"] + f * dev[k]
            u["sxy"] = f * u["sxy"]

    def state(self):
        z = torch.zeros_like(self.u[0]["vx"])
        return torch.stack([a for u in self.u for a in
                            (u["vx"], u["vy"], z, u["sxx"], u["syy"], u["szz"], u["sxy"], z, z, u["lam"], u["gam"])])

    def flux(self, d):
        out = []
        for s, r in ((0, 1.0), (1, -1.0 if d else 1.0)):
            (vn, sn), (vt, st) = self.F[d][s]
            z = torch.zeros_like(vn)
            f0, f2, f1, f4, f3 = (-r * sn / self.rho, -r * st / self.rho, -r * vn * (self.lame + 2 * self.G),
                                  -r * vn * self.lame, -r * vt * self.G)
            out += [f0, f2, z, f1, f4, f4, f3, z, z, z, z] if d == 0 else [f2, f0, z, f4, f1, f4, f3, z, z, z, z]
        return torch.stack(out)
