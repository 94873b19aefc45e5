"""The search on cell grids of chosen sizes: a small body with one particle
far from it, so that the grid of the bounding box has few particles and many
cells."""
import numpy as np
import pytest

from conftest import deck_dir, load_pkg

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
