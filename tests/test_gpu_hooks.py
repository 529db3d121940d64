"""GPU parity per hook: every C-ABI hook (include/erfx.h) against the oracle's
restatement of the same ERF function, from identical inputs.

The inputs are a mid-run state: the oracle advances one step (so every
integrator buffer holds realistic data), then every buffer is copied into the
sim, and the hook runs on both.  With the EOS on the shared reproducible pow
and no FMA contraction on either side, the bar is bit-for-bit identity of
every buffer, ghost cells included (index and ghost-cell fills exact).
"""
import ctypes

import numpy as np
import pytest

from erf_amd import config as C, problems as P
from helpers import ALL_IDS, valid
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


def _setup(kind):
    import torch
    assert torch.cuda.is_available()
    from erf_amd.lib import Sim
    if kind == "thermal":
        cfg, f = P.rising_thermal(24, 20, 16, seed=3)
        dt = 1.0
    elif kind == "cbl":
        cfg, f = P.cbl(20, 18, 16, seed=5)
        dt = 0.5
    elif kind.startswith("moist"):   # Kessler, buoyancy type moist1..moist4
        cfg, f = P.moist_bubble(24, 20, 16, seed=13, buoyancy_type=int(kind[-1]))
        dt = 1.0
    elif kind == "norain":
        cfg, f = P.moist_bubble(24, 20, 16, seed=17, norain=True)
        dt = 1.0
    elif kind.startswith("inflow"):   # ERF's Inflow on x-lo, Outflow on x-hi
        cfg, f = P.inflow_outflow(24, 16, 16, seed=19, moist=(kind == "inflow_moist"))
        if kind == "inflow_diff":     # with Constant molecular diffusion
            cfg.molec_diff_type = C.MOLEC_CONSTANT
            cfg.dynamic_viscosity, cfg.alpha_T, cfg.alpha_C = 60.0, 40.0, 50.0
        dt = 1.0
    elif kind == "noslip":   # no-slip walls, the top moving; Constant diffusion
        cfg, f = P.rising_thermal(24, 16, 16, seed=29, adv=C.ADV_UPWIND3)
        cfg.bc[2] = cfg.bc[5] = C.BC_NO_SLIP_WALL
        cfg.wall_velocity[5][0], cfg.wall_velocity[5][1] = 3.0, -1.5
        cfg.molec_diff_type = C.MOLEC_CONSTANT
        cfg.dynamic_viscosity, cfg.alpha_T = 40.0, 20.0
        dt = 1.0
    elif kind.startswith("hill"):   # terrain-following grid over a Gaussian hill
        adv = C.ADV_CENTERED2 if kind == "hill_c2" else C.ADV_UPWIND3
        cfg, f = P.hill_flow(24, 20, 16, seed=7, adv=adv, moist=(kind == "hill_moist"))
        if kind == "hill_diff":       # ConstantAlpha molecular diffusion on the terrain grid
            cfg.molec_diff_type = C.MOLEC_CONSTANT_ALPHA
            cfg.rho0_trans, cfg.dynamic_viscosity, cfg.alpha_T, cfg.alpha_C = 1.0, 60.0, 45.0, 30.0
        elif kind == "hill_noslip":   # Constant diffusion, no-slip walls, the top moving
            cfg.bc[2] = cfg.bc[5] = C.BC_NO_SLIP_WALL
            cfg.wall_velocity[5][0], cfg.wall_velocity[5][1] = 3.0, -1.5
            cfg.molec_diff_type = C.MOLEC_CONSTANT
            cfg.dynamic_viscosity, cfg.alpha_T, cfg.alpha_C = 40.0, 20.0, 10.0
        dt = 1.0
    else:  # walls + molecular diffusion
        cfg, f = P.rising_thermal(24, 8, 16, seed=11, adv=C.ADV_UPWIND3)
        cfg.bc[0] = C.BC_SYMMETRY
        cfg.bc[3] = C.BC_OUTFLOW
        cfg.molec_diff_type = C.MOLEC_CONSTANT_ALPHA
        cfg.dynamic_viscosity = 75.0
        cfg.alpha_T = 75.0
        dt = 1.0
    orc = Oracle(cfg)
    orc.load(f)
    orc.step(0.0, dt, 1)
    sim = Sim(cfg)
    ids = list(ALL_IDS) + ([C.D_EDDY] if cfg.les_type != C.LES_NONE else [])
    ids += [C.D_RAIN_ACCUM] if cfg.moisture_type != C.MOIST_NONE else []
    ids += TERRAIN_IDS if cfg.use_terrain else []
    for fid in ids:
        sim.upload(fid, orc.get(fid))
    return cfg, orc, sim, ids, dt


def _same(sim, orc, ids):
    """ids whose buffers differ anywhere (NaN == NaN), with the count of points."""
    bad = {}
    for fid in ids:
        a = sim.download(fid)
        b = orc.get(fid)
        eq = (a == b) | (np.isnan(a) & np.isnan(b))
        if not eq.all():
            d = np.abs(np.where(eq, 0.0, a - b))
            bad[fid] = (int((~eq).sum()), float(np.nanmax(d)))
    return bad


def _st(sim, s):
    return ctypes.byref(sim.state(s))


TERRAIN_IDS = [C.F_Z_ND, C.D_DETJ, C.D_AX, C.D_AY, C.D_AZ, C.D_Z_CC]
HILLS = ["hill", "hill_c2", "hill_moist", "hill_diff", "hill_noslip"]
KINDS = ["thermal", "cbl", "walls", "moist1", "moist2", "norain", "inflow", "inflow_moist", "inflow_diff",
         "noslip"] + HILLS
MOIST_BUOYANCY = ["moist1", "moist2", "moist3", "moist4"]


@pytest.mark.parametrize("kind", KINDS)
def test_cons_to_prim(kind):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, dt = _setup(kind)
    ng = sim.L.ng
    sid = C.state_id(C.S_NEW, 0)
    orc.call("orc_cons_to_prim", sid, ng)
    check(lib().erfx_cons_to_prim(sim.ctx, sim.ptr(sid), sim.ptr(C.D_PRIM), sim.ptr(C.D_PI_STAGE), ng))
    sim.sync()
    assert _same(sim, orc, ids) == {}


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("which,fast_only,synced", [(C.S_SUM, 1, 0), (C.S_NEW, 0, 0), (C.S_OLD, 0, 1)])
def test_apply_bcs(kind, which, fast_only, synced):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, dt = _setup(kind)
    ngc, ngv = (1, 1) if fast_only else (sim.L.ng, sim.L.ng - 1)
    orc.call("orc_apply_bcs", which, ngc, ngv, fast_only, synced)
    check(lib().erfx_apply_bcs(sim.ctx, _st(sim, which), sim.ptr(C.F_XVEL), sim.ptr(C.F_YVEL),
                               sim.ptr(C.F_ZVEL), ngc, ngv, fast_only, synced))
    sim.sync()
    assert _same(sim, orc, ids) == {}


# The open axis of a box: its lo and hi faces, with the other lateral axis
# periodic.  (Inflow and symmetry on x are among KINDS.)
LATERAL = {"x_slip": (0, C.BC_SLIP_WALL, C.BC_SLIP_WALL), "x_noslip": (0, C.BC_NO_SLIP_WALL, C.BC_SLIP_WALL),
           "y_slip": (1, C.BC_SLIP_WALL, C.BC_SLIP_WALL), "y_noslip": (1, C.BC_SLIP_WALL, C.BC_NO_SLIP_WALL),
           "y_symmetry": (1, C.BC_SYMMETRY, C.BC_OUTFLOW), "y_outflow": (1, C.BC_OUTFLOW, C.BC_SYMMETRY),
           "y_inflow": (1, C.BC_INFLOW, C.BC_OUTFLOW), "y_inflow_moist": (1, C.BC_INFLOW, C.BC_OUTFLOW)}


def _lateral(kind, shape):
    """A box with rules on one lateral axis, in a wind oblique to its faces."""
    d, lo, hi = LATERAL[kind]
    moist = kind.endswith("moist")
    cfg, f = (P.moist_bubble if moist else P.rising_thermal)(*shape, seed=53, adv=C.ADV_UPWIND3)
    cfg.bc[d], cfg.bc[d + 3] = lo, hi
    for o in (d, d + 3):
        if cfg.bc[o] == C.BC_NO_SLIP_WALL:      # moving along itself
            cfg.wall_velocity[o][1 - d], cfg.wall_velocity[o][2] = 2.5, 0.0
        if cfg.bc[o] == C.BC_INFLOW:
            cfg.inflow_velocity[o][d], cfg.inflow_velocity[o][1 - d] = 6.0, 1.5
            cfg.inflow_density[o], cfg.inflow_theta[o], cfg.inflow_scalar[o] = 1.1, 300.0, 0.5
            if moist:
                cfg.inflow_qv[o] = 5.0e-3
    L = C.layout_for(cfg)
    ng = L.ng
    for fid, c in ((C.F_XVEL, 0), (C.F_YVEL, 1)):
        f[fid][0][ng:ng + cfg.nz, ng:ng + cfg.ny + c, ng:ng + cfg.nx + 1 - c] += 6.0 if c == d else 1.5
    return cfg, f


def _fill(sim, orc, which, ngc, ngv, fast_only, synced):
    from erf_amd.lib import lib, check
    orc.call("orc_apply_bcs", which, ngc, ngv, fast_only, synced)
    check(lib().erfx_apply_bcs(sim.ctx, _st(sim, which), sim.ptr(C.F_XVEL), sim.ptr(C.F_YVEL),
                               sim.ptr(C.F_ZVEL), ngc, ngv, fast_only, synced))
    sim.sync()


@pytest.mark.parametrize("kind", list(LATERAL))
@pytest.mark.parametrize("shape", [(20, 18, 16), (9, 67, 8), (70, 7, 9)])
def test_lateral_rules(kind, shape):
    """Rules on the faces of one lateral axis, x or y: every fill (narrow and at full
    width, fast variables alone and all, synced) and whole steps against the
    oracle, bit for bit."""
    import torch
    assert torch.cuda.is_available()
    from erf_amd.lib import Sim
    cfg, f = _lateral(kind, shape)
    orc, sim = Oracle(cfg), Sim(cfg)
    orc.load(f)
    orc.step(0.0, 0.5, 1)
    ids = list(ALL_IDS) + ([C.D_RAIN_ACCUM] if cfg.moisture_type != C.MOIST_NONE else [])
    for fid in ids:
        sim.upload(fid, orc.get(fid))
    ng = sim.L.ng
    for args in ((C.S_SUM, 1, 1, 1, 0), (C.S_SUM, 2, 1, 0, 0), (C.S_SUM, ng, ng - 1, 1, 0),
                 (C.S_NEW, ng, ng - 1, 0, 0), (C.S_OLD, ng, ng - 1, 0, 1)):
        _fill(sim, orc, *args)
        assert _same(sim, orc, ids) == {}, args
    orc, sim = Oracle(cfg), Sim(cfg)
    orc.load(f)
    sim.load(f)
    orc.step(0.0, 0.5, 3)
    sim.step(0.0, 0.5, 3)
    for fid in (C.F_CONS, C.F_XVEL, C.F_YVEL, C.F_ZVEL):
        a, b = (valid(x.get(fid) if x is orc else x.download(fid), cfg, x.L, fid) for x in (sim, orc))
        assert np.array_equal(a, b), fid


@pytest.mark.parametrize("kind", ["thermal", "moist1", "walls", "inflow", "inflow_moist", "noslip", "hill"])
def test_apply_bcs_fast_only_full_width(kind):
    """the fill between substeps that are not chained: the fast variables at the full
    velocity width; and with the ghost widths apart"""
    cfg, orc, sim, ids, dt = _setup(kind)
    ng = sim.L.ng
    for ngc, ngv in ((ng, ng - 1), (1, ng - 1), (ng, 1)):
        _fill(sim, orc, C.S_SUM, ngc, ngv, 1, 0)
        assert _same(sim, orc, ids) == {}, (ngc, ngv)


@pytest.mark.parametrize("kind", ["thermal", "inflow", "hill"])
@pytest.mark.parametrize("shape", [(4, 4, 8), (5, 7, 8), (67, 6, 9), (8, 33, 17)])
def test_apply_bcs_small_and_ragged(kind, shape):
    """The launch around the box leaves out a core 1 .. n-2: boxes whose core is
    two cells wide, ones that wrap several columns per work-group, odd sizes."""
    from erf_amd.lib import Sim, lib, check
    make = {"thermal": P.rising_thermal, "inflow": P.inflow_outflow, "hill": P.hill_flow}[kind]
    cfg, f = make(*shape, seed=31)
    orc = Oracle(cfg)
    orc.load(f)
    orc.step(0.0, 0.5, 1)
    sim = Sim(cfg)
    ids = list(ALL_IDS) + (TERRAIN_IDS if cfg.use_terrain else [])
    for fid in ids:
        sim.upload(fid, orc.get(fid))
    ng = sim.L.ng
    for which, synced in ((C.S_NEW, 0), (C.S_OLD, 1)):
        orc.call("orc_apply_bcs", which, ng, ng - 1, 0, synced)
        check(lib().erfx_apply_bcs(sim.ctx, _st(sim, which), sim.ptr(C.F_XVEL), sim.ptr(C.F_YVEL),
                                   sim.ptr(C.F_ZVEL), ng, ng - 1, 0, synced))
    sim.sync()
    assert _same(sim, orc, ids) == {}
    orc, sim = Oracle(cfg), Sim(cfg)
    orc.load(f)
    sim.load(f)
    orc.step(0.0, 0.5, 3)
    sim.step(0.0, 0.5, 3)
    for fid in (C.F_CONS, C.F_XVEL, C.F_YVEL, C.F_ZVEL):
        a, b = (valid(x.get(fid) if x is orc else x.download(fid), cfg, x.L, fid) for x in (sim, orc))
        assert np.array_equal(a, b), fid


@pytest.mark.parametrize("kind", KINDS)
def test_make_fast_coeffs(kind):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, dt = _setup(kind)
    dtau = dt / cfg.mri_ratio
    orc.call("orc_make_fast_coeffs", dtau, 0.1)
    check(lib().erfx_make_fast_coeffs(sim.ctx, sim.ptr(C.D_FAST_COEFFS), _st(sim, C.S_NEW), sim.ptr(C.D_PRIM),
                                      sim.ptr(C.D_PI_STAGE), dtau, 0.1))
    sim.sync()
    assert _same(sim, orc, ids) == {}


@pytest.mark.parametrize("kind", ["dry", "moist", "hill", "hill_moist"])
@pytest.mark.parametrize("shape", [(64, 64, 128), (96, 96, 40), (97, 95, 64), (96, 96, 65), (128, 128, 9),
                                   (129, 128, 9)])
def test_make_fast_coeffs_forms(kind, shape):
    """Each form by box size: 16-column tiles with the most levels they take,
    32-column tiles (three and four levels per chunk, the last tile partial, the
    largest column count), one lane per column past the tiles' levels and past their
    columns.  All five components bit-identical to the oracle's from the same state
    (one step on the GPU)."""
    import torch
    assert torch.cuda.is_available()
    from erf_amd.lib import Sim, lib, check
    make = {"dry": P.rising_thermal, "moist": P.moist_bubble}.get(kind)
    cfg, f = make(*shape, seed=47) if make else P.hill_flow(*shape, seed=47, moist=(kind == "hill_moist"))
    sim, orc = Sim(cfg), Oracle(cfg)
    sim.load(f)
    orc.load(f)
    sim.step(0.0, 0.2, 1)
    for fid in [C.state_id(C.S_NEW, 0), C.D_PRIM, C.D_PI_STAGE, C.F_R0, C.F_P0, C.F_PI0, C.D_FAST_COEFFS]:
        orc.set(fid, sim.download(fid))
    orc.call("orc_make_fast_coeffs", 0.05, 0.1)
    check(lib().erfx_make_fast_coeffs(sim.ctx, sim.ptr(C.D_FAST_COEFFS), _st(sim, C.S_NEW), sim.ptr(C.D_PRIM),
                                      sim.ptr(C.D_PI_STAGE), 0.05, 0.1))
    sim.sync()
    a, b = sim.download(C.D_FAST_COEFFS), orc.get(C.D_FAST_COEFFS)
    assert np.array_equal(a, b, equal_nan=True), [int((x != y).sum()) for x, y in zip(a, b)]
    assert np.abs(valid(b, cfg, sim.L, C.D_FAST_COEFFS)[1]).min() > 0.0


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("step,nrk", [(0, 0), (0, 2), (3, 2)])
def test_fast_rhs_N(kind, step, nrk):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, dt = _setup(kind)
    dtau = dt / cfg.mri_ratio
    nsub = cfg.mri_ratio
    beta_s = 0.1 if cfg.implicit_substepping else -1.0
    T = "T" if cfg.use_terrain else "N"       # erf_fast_rhs_T on a terrain grid
    orc.call("orc_fast_rhs_" + T, step, nrk, dtau, beta_s, 1.0 / nsub)
    prev = C.S_OLD if step == 0 else C.S_SUM
    check(getattr(lib(), "erfx_fast_rhs_" + T)(sim.ctx, step, nrk, _st(sim, C.F_SLOW), _st(sim, prev), _st(sim, C.S_NEW),
                                sim.ptr(C.D_PRIM), sim.ptr(C.D_PI_STAGE), sim.ptr(C.D_FAST_COEFFS),
                                _st(sim, C.S_SUM), _st(sim, C.S_SCRATCH), dtau, beta_s, 1.0 / nsub))
    sim.sync()
    assert _same(sim, orc, ids) == {}


@pytest.mark.parametrize("kind", ["cbl"])
def test_turbulent_viscosity(kind):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, dt = _setup(kind)
    orc.call("orc_turbulent_viscosity")
    check(lib().erfx_turbulent_viscosity(sim.ctx, sim.ptr(C.state_id(C.S_OLD, 0)), sim.ptr(C.D_XVEL_OLD),
                                         sim.ptr(C.D_YVEL_OLD), sim.ptr(C.D_ZVEL_OLD), sim.ptr(C.D_EDDY), None))
    sim.sync()
    assert _same(sim, orc, ids) == {}


@pytest.mark.parametrize("kind", KINDS + ["moist3", "moist4"])
@pytest.mark.parametrize("nrk", [0, 2])
def test_slow_rhs_pre(kind, nrk):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, dt = _setup(kind)
    slow_dt = dt / 3.0 if nrk == 0 else dt
    orc.call("orc_slow_rhs_pre", nrk, slow_dt)
    eddy = sim.ptr(C.D_EDDY) if cfg.les_type != C.LES_NONE else None
    check(lib().erfx_slow_rhs_pre(sim.ctx, nrk, slow_dt, _st(sim, C.F_SLOW), _st(sim, C.S_NEW), sim.ptr(C.D_PRIM),
                                  _st(sim, C.S_SCRATCH), sim.ptr(C.F_XVEL), sim.ptr(C.F_YVEL), sim.ptr(C.F_ZVEL),
                                  eddy, None))
    sim.sync()
    assert _same(sim, orc, ids) == {}


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nrk", [0, 2])
def test_slow_rhs_post(kind, nrk):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, dt = _setup(kind)
    slow_dt = dt / 3.0 if nrk == 0 else dt
    orc.call("orc_slow_rhs_post", nrk, slow_dt)
    eddy = sim.ptr(C.D_EDDY) if cfg.les_type != C.LES_NONE else None
    check(lib().erfx_slow_rhs_post(sim.ctx, nrk, slow_dt, _st(sim, C.F_SLOW), _st(sim, C.S_OLD), _st(sim, C.S_NEW),
                                   _st(sim, C.S_SUM), sim.ptr(C.D_PRIM), _st(sim, C.S_SCRATCH), sim.ptr(C.F_XVEL),
                                   sim.ptr(C.F_YVEL), eddy))
    sim.sync()
    assert _same(sim, orc, ids) == {}


@pytest.mark.parametrize("kind", ["moist1", "norain", "hill_moist"])
@pytest.mark.parametrize("dt", [1.0, 3.0])
def test_kessler(kind, dt):
    from erf_amd.lib import lib, check
    cfg, orc, sim, ids, _ = _setup(kind)
    orc.kessler(dt)
    check(lib().erfx_kessler_advance(sim.ctx, sim.ptr(C.F_CONS), dt, sim.ptr(C.D_RAIN_ACCUM)))
    assert _same(sim, orc, ids) == {}


@pytest.mark.parametrize("h0", [0.0, 500.0])
def test_terrain_metrics(h0):
    """make_J / make_areas / make_zcc from uploaded node heights (the whole
    layout, padding included) and the dz_min of the time-step estimate."""
    import torch
    assert torch.cuda.is_available()
    from erf_amd.lib import Sim
    cfg, f = P.hill_flow(24, 20, 16, h0=h0)
    orc = Oracle(cfg)
    orc.load(f)
    sim = Sim(cfg)
    sim.upload(C.F_Z_ND, f[C.F_Z_ND])
    assert _same(sim, orc, TERRAIN_IDS) == {}


def test_fast_rhs_N_rejects_terrain():
    from erf_amd.lib import lib
    cfg, orc, sim, ids, dt = _setup("hill")
    rc = lib().erfx_fast_rhs_N(sim.ctx, 0, 0, _st(sim, C.F_SLOW), _st(sim, C.S_OLD), _st(sim, C.S_NEW),
                               sim.ptr(C.D_PRIM), sim.ptr(C.D_PI_STAGE), sim.ptr(C.D_FAST_COEFFS),
                               _st(sim, C.S_SUM), _st(sim, C.S_SCRATCH), 1.0 / 6, 0.1, 1.0)
    assert rc != 0


def _substep(sim, prev, step, beta_s):
    from erf_amd.lib import lib, check
    check(lib().erfx_fast_rhs_N(sim.ctx, step, 2, _st(sim, C.F_SLOW), _st(sim, prev), _st(sim, C.S_NEW),
                                sim.ptr(C.D_PRIM), sim.ptr(C.D_PI_STAGE), sim.ptr(C.D_FAST_COEFFS),
                                _st(sim, C.S_SUM), _st(sim, C.S_SCRATCH), 0.05, beta_s, 0.2))


@pytest.mark.parametrize("moist", [False, True])
@pytest.mark.parametrize("shape", [(24, 20, 9), (41, 23, 128), (96, 96, 7), (97, 95, 13), (96, 96, 31), (96, 96, 40), (97, 95, 65), (96, 96, 97)])
@pytest.mark.parametrize("implicit,separate", [(True, True), (False, False), (False, True)])
def test_substep_tiles_separate_and_explicit(shape, moist, implicit, separate):
    """The substep whose state is not the one it reads (S_prev and S_data in
    buffers of their own after the first substep, with other densities in the
    two) and the explicit one: the tile form, in each of its chunk sizes, against one
    lane per column, bit for bit."""
    import torch
    assert torch.cuda.is_available()
    from erf_amd.lib import Sim
    cfg, f = (P.moist_bubble if moist else P.rising_thermal)(*shape, seed=37, adv=C.ADV_UPWIND3)
    cfg.implicit_substepping = int(implicit)
    out = []
    for variant in (C.COL_VARIANTS - 1, 7):        # tiles, one lane per column
        sim = Sim(cfg)
        sim.load(f)
        sim.step(0.0, 0.1, 1)
        sim.set_column_variant(variant)
        _substep(sim, C.S_OLD if separate else C.S_SUM, 1, 0.1 if implicit else -1.0)
        sim.sync()
        out.append([sim.download(C.state_id(s, c)) for s in (C.S_SUM, C.S_SCRATCH) for c in range(4)])
        sim.close()
    for n, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b, equal_nan=True), n


@pytest.mark.parametrize("shape,implicit,separate,share",
                         [((64, 64, 64), True, False, 0.5), ((64, 64, 64), True, True, 0.5),
                          ((64, 64, 64), False, False, 0.5), ((512, 128, 4), True, False, 1.25)])
def test_substep_tiles_run(shape, implicit, separate, share):
    """The tile form runs where it is the faster one.  64 x 64 x 64, in place and
    in separate buffers, implicit and explicit: a third of one lane per column's
    time (28 us and 92 us a substep); half is asked for.  Few levels on many
    columns: 23 us and 27 us; a quarter more than 27 is asked for (tiles of fewer
    columns, most of whose lanes idle there, take 44)."""
    import time
    import torch
    assert torch.cuda.is_available()
    from erf_amd.lib import Sim
    cfg, f = P.rising_thermal(*shape, seed=41, adv=C.ADV_UPWIND3)
    cfg.implicit_substepping = int(implicit)
    sim = Sim(cfg)
    sim.load(f)
    sim.step(0.0, 0.1, 1)
    took = {}
    for variant in (C.COL_VARIANTS - 1, 7):
        sim.set_column_variant(variant)
        best = []
        for _ in range(5):
            sim.sync()
            t = time.perf_counter()
            for _ in range(40):
                _substep(sim, C.S_OLD if separate else C.S_SUM, 1, 0.1 if implicit else -1.0)
            sim.sync()
            best.append(time.perf_counter() - t)
        took[variant] = min(best)
    sim.close()
    assert took[C.COL_VARIANTS - 1] < share * took[7], took
