"""Tiles of the pair kernels at the sizes where their cutting can go wrong,
against the oracle, every state field and the pair list bit for bit.

The receivers of a tile come from one strip of the cell grid; a body of fewer
cells than a strip, a last strip one cell wide, strips that fill their tiles
exactly or by one particle over, strips of a low body (more strips than the
tile capacity, which falls back to tiles cut every TILE slots) and particles
outside the domain box are the edges.
"""
import dataclasses
import importlib

import numpy as np
import pytest

from conftest import ORACLE_LIB, bits_equal, deck_dir, describe_diff, load_pkg

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vel", "stress", "internal_vars", "f_drucker", "displ", "grad_u", "ddev_strn", "f_bound", "art_visc",
          "if_out_domain")

# name: (deck, lattice columns, rows, smoothing factor, other changes)
BODIES = {
    "one_particle_row_strip": ("c1_collapse", 21, 2, 1.2, {}),
    "narrower_than_a_strip": ("c1_collapse", 7, 120, 1.2, {}),
    "last_strip_one_cell": ("c1_collapse", 21, 90, 1.2, {}),
    "full_tiles": ("c1_collapse", 64, 64, 1.0, {}),           # 16 columns a strip: 4 tiles exactly
    "one_over": ("c1_collapse", 65, 65, 1.0, {}),
    "low_body_many_strips": ("c1_collapse", 400, 4, 0.5, {}),  # falls back: cells one spacing wide
    "cspm_moving": ("t2_cspm", 50, 37, 1.2, {}),
    "xsph_two_points": ("t4_xsph", 43, 31, 1.2, {"npoints": 2}),
    "four_points": ("t5_sp4", 37, 41, 1.2, {}),
    "four_points_xsph": ("t5_sp4", 30, 30, 1.2, {"xsph": True}),
}


def body(name):
    sps = load_pkg()
    deck_name, nx, ny, sml, change = BODIES[name]
    deck = dataclasses.replace(sps.read_deck(deck_dir(deck_name)), sml=sml, **change)
    dx = deck.dx
    # the lattice counts are int(length / dx + 1): half a spacing beyond the last column
    deck.xs = (0.0, (nx - 0.5) * dx, 0.0, (nx - 0.5) * dx)
    deck.ys = (0.0, 0.0, (ny - 0.5) * dx, (ny - 0.5) * dx)
    deck.dy = dx
    if name == "low_body_many_strips":   # the box close around the body
        deck.xmin_domain = np.array([-8 * dx, -8 * dx])
        deck.xmax_domain = np.array([(nx + 4) * dx, (ny + 8) * dx])
        deck.dummy_nodes, deck.walls = False, []
    return sps, deck


def compare(gpu, ora, what):
    g, o = gpu.get_state(), ora.get_state()
    bad = [f"{k}: {describe_diff(o[k], g[k])}" for k in FIELDS if not bits_equal(o[k], g[k])]
    p, q = gpu.get_pairs(), ora.get_pairs()
    bad += [f"pairs.{k}" for k in p if not bits_equal(q[k], p[k])]
    assert not bad, f"{what}: " + "; ".join(bad)


@pytest.mark.parametrize("name", sorted(BODIES))
def test_tiles_against_oracle(name):
    sps, deck = body(name)
    gpu = sps.Simulation.from_deck(deck)
    ora = sps.Simulation.from_deck(deck, lib_path=ORACLE_LIB)
    print(f"[tiles] {name}: {gpu.n2} particles", flush=True)
    # a moving start: pair counts rise and fall, so pairs lie on both sides of
    # the list's high-water mark; a few particles start outside the domain box
    rng = np.random.default_rng(11)
    st = sps.initial_state(gpu.parts, gpu.niv)
    st["vel"][:gpu.n] = 2.0 * rng.standard_normal((gpu.n, 2))
    for k in (3, gpu.nn + 5):
        st["x"][k] = deck.xmax_domain + 10.0 * deck.dx
    for sim in (gpu, ora):
        sim.set_state(st)
    for step in range(1, 7):
        gpu.step(1)
        ora.step(1)
        compare(gpu, ora, f"{name} step {step}")


# The mixed form cuts its tiles every TILE slots: bodies where few, many and
# all tiles cross a strip end and read their lists by storage slot.  An
# elastic deck from rest, so the difference to the double-precision oracle is
# the rounding of the pair terms: each of about 20 terms of a sum to 2^-24 of
# itself, compensated; with the smallest sums two orders below their terms,
# 20 steps stay under 1e-5 of the largest value.
@pytest.mark.parametrize("skin", [0.0, 0.25])
@pytest.mark.parametrize("nx,ny,change", [(17, 16, {}), (65, 65, {}), (200, 5, {}), (33, 90, {"xsph": True}),
                                          (40, 40, {"npoints": 2})])
def test_mixed_tiles_across_strips(nx, ny, change, skin):
    sps = load_pkg()
    acc = importlib.import_module("stress-particle-sph_amd.accuracy")
    deck = dataclasses.replace(sps.read_deck(deck_dir("t3_elastic")), **change)
    deck.xs = (0.0, (nx - 0.5) * deck.dx, 0.0, (nx - 0.5) * deck.dx)
    deck.ys = (0.0, 0.0, (ny - 0.5) * deck.dx, (ny - 0.5) * deck.dx)
    mix = sps.Simulation.from_deck(deck, mode=sps.MODE_FAST)
    if skin:
        mix.set_list_skin(skin * deck.dx)
    ora = sps.Simulation.from_deck(deck, lib_path=ORACLE_LIB)
    x0 = ora.get_state(["x"])["x"]
    print(f"[tiles] mixed {nx} x {ny} {change} skin {skin}", flush=True)
    mix.step(20)
    ora.step(20)
    err = acc.compare_states(mix.get_state(), ora.get_state(), x0)
    for k in ("disp_rel_max", "vel_rel_max", "stress_rel_max"):
        assert err[k] <= 1e-5, f"{k} {err[k]:.3e}"


# The search's prefix sums run over 3 (cells + 1) + 1 buckets and over the
# cells, 2048 elements a tile: one particle far from the body stretches the
# grid to a few cells under and over a tile, over the 64 tiles that one look
# back takes and over the 1024 blocks of a launch.
@pytest.mark.parametrize("cells", [100, 681, 682, 683, 2047, 2048, 45000, 800000])
def test_search_on_stretched_grids(cells):
    sps = load_pkg()
    deck = sps.read_deck(deck_dir("t1_tiny"))
    reach = 2 * 1.2 * deck.dx
    side = max(1.0, np.sqrt(cells))
    deck.xmax_domain = np.array([side + 40.0, cells / side + 40.0]) * reach
    gpu = sps.Simulation.from_deck(deck)
    ora = sps.Simulation.from_deck(deck, lib_path=ORACLE_LIB)
    st = sps.initial_state(gpu.parts, gpu.niv)
    st["x"][gpu.nn - 1] = np.array([side - 0.5, cells / side - 0.5]) * reach
    for sim in (gpu, ora):
        sim.set_state(st)
    print(f"[search] about {cells} cells", flush=True)
    for step in range(1, 4):
        gpu.step(1)
        ora.step(1)
        compare(gpu, ora, f"{cells} cells, step {step}")


# The free surface: four lanes share a particle's pairs in list order.  Few and
# many partners (over the 96 held in LDS, over 32 of a kind in a cell: then a
# lane walks them all), particles on both sides of the list's high-water mark,
# a body of fewer particles than a block.
@pytest.mark.parametrize("deck_name,nx,ny,change", [
    ("c1_collapse", 5, 3, {}), ("c1_collapse", 65, 33, {}), ("c1_collapse", 40, 40, {"sml": 2.4}),
    ("c1_collapse", 40, 30, {"sml": 3.4}), ("t5_sp4", 30, 30, {}), ("t4_xsph", 33, 47, {"npoints": 2})])
def test_surface_against_oracle(deck_name, nx, ny, change):
    sps = load_pkg()
    deck = dataclasses.replace(sps.read_deck(deck_dir(deck_name)), **change)
    deck.xs = (0.0, (nx - 0.5) * deck.dx, 0.0, (nx - 0.5) * deck.dx)
    deck.ys = (0.0, 0.0, (ny - 0.5) * deck.dx, (ny - 0.5) * deck.dx)
    deck.dy = deck.dx
    gpu = sps.Simulation.from_deck(deck)
    ora = sps.Simulation.from_deck(deck, lib_path=ORACLE_LIB)
    st = sps.initial_state(gpu.parts, gpu.niv)
    st["vel"][:gpu.n] = 2.0 * np.random.default_rng(3).standard_normal((gpu.n, 2))
    for sim in (gpu, ora):
        sim.set_state(st)
    print(f"[surface] {deck_name} {nx} x {ny} {change}", flush=True)
    for step in range(1, 5):
        gpu.step(1)
        ora.step(1)
        for what, a, b in zip(("bc_or_not", "normal"), ora.get_surface(), gpu.get_surface()):
            assert bits_equal(a, b), f"step {step}: {what}"
