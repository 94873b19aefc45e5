"""The search on cell grids of chosen sizes: a small body with one particle
far from it, so that the grid of the bounding box has few particles and many
cells."""
import numpy as np
import pytest

from conftest import ORACLE_LIB, deck_dir, load_pkg
from test_gpu_tiles import compare

pytestmark = pytest.mark.gpu


def stretched(sps, ndivx, ndivy, **kw):
    """The smallest deck on a grid of ndivx x ndivy cells (2h wide), with its
    state; the far particle sits in the last cell."""
    deck = sps.read_deck(deck_dir("t1_tiny"))
    cell = 2 * 1.2 * deck.dx
    deck.xmax_domain = np.array([ndivx + 40.0, ndivy + 40.0]) * cell
    sim = sps.Simulation.from_deck(deck, **kw)
    st = sps.initial_state(sim.parts, sim.niv)
    lo = st["x"].min(axis=0)
    st["x"][sim.nn - 1] = lo + np.array([ndivx - 0.5, ndivy - 0.5]) * cell
    sim.set_state(st)
    return sim


# What a search does per particle may not take longer because the grid has many
# cells: a launch of three blocks that clears 2.4 million counters took sixty times
# as long as on the small grid.  Event times of a launch are 6 us at least.
def test_per_particle_passes_on_a_wide_grid():
    sps = load_pkg()
    ms = {}
    for cells in (60, 900):
        sim = stretched(sps, cells, cells)
        print(f"[grids] {cells} x {cells}", flush=True)
        sim.step(2)
        sim.set_profiling(True)
        sim.step(10)
        ms[cells] = {k: t / n for k, (n, t) in sim.profile().items()}
        st = sim.stats()
        assert (st["ndivx"], st["ndivy"]) == (cells, cells)
        sim.close()
    for k in ("k_permute", "k_cell_count", "k_cell_scatter"):
        assert ms[900][k] <= 4 * ms[60][k], f"{k}: {1e3 * ms[60][k]:.1f} us on 60 x 60, {1e3 * ms[900][k]:.1f} us on 900 x 900"


# The scans of a search read the bucket counts and write their prefixes, read
# those for the cells' totals and write theirs: 40 bytes a cell.  At 1 TB/s, an
# eighth of the memory's rate, 8.4 M cells take 336 us.
def test_scan_rate_on_a_wide_grid():
    sps = load_pkg()
    sim = stretched(sps, 2900, 2900)
    print("[grids] 2900 x 2900", flush=True)
    sim.step(2)
    sim.set_profiling(True)
    sim.step(10)
    us = 1e3 * sim.profile()["k_scan"][1] / 10
    assert us <= 2900 * 2900 * 40 / 1e6, f"{us:.0f} us of scans a search"


# The search scans 3 (cells + 1) + 1 bucket counts, 4096 a tile, and cells + 1
# totals, 1024 a tile: one tile and the next, the 64 tiles of one look back and
# the next, the 1024 runs of a launch and more tiles than runs (then a run has
# two or more), each at its last full count and around it.
GRIDS = [(31, 33), (14, 73), (32, 32),                  # 1024 cell totals, one fewer, one more
         (29, 47), (31, 44), (15, 91),                  # 4093, 4096 and 4099 buckets
         (255, 257), (256, 256),                        # 64 tiles of cells, 65
         (340, 257), (399, 219),                        # 64 tiles of buckets, 65
         (1023, 1025), (1024, 1024),                    # 1024 runs of cells; 513 of two tiles
         (1100, 1271), (1182, 1183),                    # 1024 runs of buckets; 513 of two tiles
         (2100, 2001), (3001, 2003)]                    # five and six tiles of cells a run


@pytest.mark.parametrize("ndivx,ndivy", GRIDS)
def test_scans_against_oracle(ndivx, ndivy):
    sps = load_pkg()
    gpu, ora = stretched(sps, ndivx, ndivy), stretched(sps, ndivx, ndivy, lib_path=ORACLE_LIB)
    print(f"[grids] {ndivx} x {ndivy}", flush=True)
    for step in range(1, 4):                            # later scans in the words of the earlier ones
        gpu.step(1)
        ora.step(1)
        compare(gpu, ora, f"{ndivx} x {ndivy}, step {step}")
    st = gpu.stats()
    assert (st["ndivx"], st["ndivy"]) == (ndivx, ndivy)
