"""Launch-level options of the sim against the plain path:

* the step sequence replayed from a captured hipGraph (erfx_sim_set_graph):
  bit-identical after every replay, with eager work and host synchronisation
  between the replays, for dry, moist (Kessler) and terrain cases; a change of
  dt re-captures the graph;
* every variant of the acoustic column kernel (erfx_sim_set_column_variant)
  and the autotuner that picks one (erfx_sim_autotune): bit-identical."""
import numpy as np
import pytest

from erf_amd import config as C, problems as P

pytestmark = pytest.mark.gpu

FIELDS = (C.F_CONS, C.F_XVEL, C.F_YVEL, C.F_ZVEL)


def _pair(cfg, f):
    import torch
    assert torch.cuda.is_available()
    from erf_amd.lib import Sim
    a, b = Sim(cfg), Sim(cfg)
    a.load(f)
    b.load(f)
    a.set_graph(True)
    return a, b


def _same(a, b):
    bad = []
    for fid in FIELDS:
        x, y = a.download(fid), b.download(fid)
        if not np.array_equal(x, y, equal_nan=True):
            bad.append(fid)
    return bad


@pytest.mark.parametrize("case", ["thermal", "moist", "hill"])
def test_graph_replay_matches_direct(case):
    if case == "thermal":
        cfg, f = P.rising_thermal(32, 24, 16, seed=5)
    elif case == "moist":
        cfg, f = P.moist_bubble(24, 20, 16, seed=7)
    else:
        cfg, f = P.hill_flow(24, 20, 16, seed=9)
    a, b = _pair(cfg, f)
    t = 0.0
    for rep in range(3):                      # three replays of the same graph
        a.step(t, 1.0, 2)
        b.step(t, 1.0, 2)
        t += 2.0
        assert _same(a, b) == [], (case, rep)
        b.download(C.F_CONS)                  # eager work between replays
    a.step(t, 1.0, 3)                         # one replay plus one direct step
    b.step(t, 1.0, 3)
    t += 3.0
    assert _same(a, b) == []
    a.step(t, 0.5, 2)                         # new dt: captured again
    b.step(t, 0.5, 2)
    assert _same(a, b) == []
    a.close()
    b.close()


@pytest.mark.parametrize("variant", list(range(C.COL_VARIANTS)))
def test_column_variants_identical(variant):
    cfg, f = P.rising_thermal(40, 24, 16, seed=11, adv=C.ADV_UPWIND3)
    a, b = _pair(cfg, f)
    a.set_graph(False)
    a.set_column_variant(variant)
    a.step(0.0, 1.0, 3)
    b.step(0.0, 1.0, 3)
    assert _same(a, b) == []
    a.close()
    b.close()


def test_autotune_picks_a_variant_and_keeps_results():
    cfg, f = P.moist_bubble(24, 20, 16, seed=13)
    a, b = _pair(cfg, f)
    a.set_graph(False)
    a.autotune(True)
    a.step(0.0, 1.0, 3)          # 3 steps x 10 substeps: each of the 10 variants timed 3 times
    b.step(0.0, 1.0, 3)
    v, ms = a.column_variant()
    assert 0 <= v < C.COL_VARIANTS and all(m > 0 for m in ms) and ms[v] == min(ms)
    a.step(3.0, 1.0, 2)          # with the chosen variant
    b.step(3.0, 1.0, 2)
    assert _same(a, b) == []
    a.close()
    b.close()


@pytest.mark.parametrize("case", ["flat37", "flat_moist_50", "hill21", "hill_moist_30", "flat_deep128",
                                  "flat_tc32_40", "flat_tc32_80", "flat_tc32_deep100"])
def test_tile_form_matches_column_form(case):
    """The tile form of the acoustic column kernel (the default) against the
    one-lane-per-column form on level counts that leave the last chunk partial and
    trailing chunks empty, flat and terrain, dry and moist: bit-identical after
    several steps.  Boxes of up to 8,160 columns take 16-column tiles (32 chunks
    of levels: one level each at 21 and 30 levels, two at 37 and 50, four at 128),
    larger ones 32-column tiles (16 chunks: three levels each at 40, five at 80,
    seven at 100)."""
    if case == "flat37":
        cfg, f = P.rising_thermal(40, 24, 37, seed=21, adv=C.ADV_UPWIND3)
    elif case == "flat_deep128":
        cfg, f = P.rising_thermal(40, 24, 128, seed=25, adv=C.ADV_UPWIND3)
    elif case.startswith("flat_tc32"):
        nz = {"flat_tc32_40": 40, "flat_tc32_80": 80, "flat_tc32_deep100": 100}[case]
        cfg, f = P.rising_thermal(96, 96, nz, seed=26, adv=C.ADV_UPWIND3)
    elif case == "flat_moist_50":
        cfg, f = P.moist_bubble(24, 20, 50, seed=22)
    elif case == "hill21":
        cfg, f = P.hill_flow(24, 20, 21, seed=23)
    else:
        cfg, f = P.hill_flow(24, 20, 30, seed=24, moist=True)
    a, b = _pair(cfg, f)
    a.set_graph(False)
    a.set_column_variant(7)          # one lane per column
    a.step(0.0, 1.0, 3)
    b.step(0.0, 1.0, 3)
    assert _same(a, b) == []
    a.close()
    b.close()


@pytest.mark.parametrize("moist", [False, True])
@pytest.mark.parametrize("shape", [(24, 20, 9), (24, 20, 33), (41, 23, 128), (96, 96, 16), (97, 95, 65), (96, 96, 97),
                                   (96, 96, 128)])
def test_tile_form_chunk_edges(shape, moist):
    """The tile form where its chunks of levels change: one level per chunk (9
    levels), two in 64-column tiles (16), one level past a full set of chunks (33 = 32 + 1 in 16-column
    tiles, 65 = 16 x 4 + 1 and 97 = 16 x 6 + 1 in 32-column tiles), the largest
    it takes (128), and a column count that leaves the last tile partial (41 x
    23, 97 x 95): bit-identical with one lane per column."""
    case = P.moist_bubble if moist else P.rising_thermal
    cfg, f = case(*shape, seed=31, adv=C.ADV_UPWIND3)
    a, b = _pair(cfg, f)
    a.set_graph(False)
    a.set_column_variant(7)          # one lane per column
    a.step(0.0, 0.5, 2)
    b.step(0.0, 0.5, 2)
    assert _same(a, b) == []
    a.close()
    b.close()


@pytest.mark.parametrize("moist", [False, True])
@pytest.mark.parametrize("shape", [(96, 96, 4), (97, 95, 8), (97, 95, 9), (96, 96, 16), (97, 95, 17), (96, 96, 32),
                                   (97, 95, 33), (91, 90, 20), (90, 90, 20)])
def test_tile_form_few_levels(shape, moist):
    """64-column tiles at the edges of their chunk sizes (one, two and four
    levels: 8, 16 and 32 levels), one level past the last, a last tile that is
    partial, the first column count that takes them and the last that does not:
    bit-identical with one lane per column.  (4 levels are below the fused fills'
    size, so there the launch carries the ghost layer as well.)"""
    case = P.moist_bubble if moist else P.rising_thermal
    cfg, f = case(*shape, seed=43, adv=C.ADV_UPWIND3)
    a, b = _pair(cfg, f)
    a.set_graph(False)
    a.set_column_variant(7)          # one lane per column
    a.step(0.0, 0.5, 2)
    b.step(0.0, 0.5, 2)
    assert _same(a, b) == []
    a.close()
    b.close()


@pytest.mark.parametrize("moist", [False, True])
@pytest.mark.parametrize("shape", [(97, 95, 65), (96, 96, 75), (96, 96, 96), (96, 96, 64), (97, 95, 97)])
def test_terrain_tile_form_chunk_edges(shape, moist):
    """The terrain grid's 32-column tiles: five levels per chunk with a last tile
    that is partial (65 levels), five and six with a last chunk that is (75), six in
    full (96), the four of the smaller form (64), and one level past what they take:
    bit-identical with one lane per column."""
    cfg, f = P.hill_flow(*shape, seed=59, moist=moist)
    a, b = _pair(cfg, f)
    a.set_graph(False)
    a.set_column_variant(7)          # one lane per column
    a.step(0.0, 0.2, 2)
    b.step(0.0, 0.2, 2)
    x = a.download(C.F_CONS)[C.RHO]
    assert np.isfinite(x).all()
    assert _same(a, b) == []
    a.close()
    b.close()
