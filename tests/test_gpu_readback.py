"""The state taken back from the device, against the arrays it was set from,
bit for bit: fields that fit one staging chunk (1 MiB), that end in the
middle of one, and that take several per thread; every field at once, some,
one, and none."""
import ctypes
import dataclasses

import numpy as np
import pytest

from conftest import bits_equal, deck_dir, load_pkg

pytestmark = pytest.mark.gpu

SUBSETS = {"all": None, "one": ["f_drucker"], "narrow": ["if_out_domain", "wall_position", "x"], "none": ["itype"]}


@pytest.mark.parametrize("nx,ny", [(5, 4), (127, 129), (256, 256), (500, 411)])
def test_state_as_set(nx, ny):
    sps = load_pkg()
    deck = sps.read_deck(deck_dir("t3_elastic"))
    deck = dataclasses.replace(deck)
    deck.xs = (0.0, (nx - 0.5) * deck.dx, 0.0, (nx - 0.5) * deck.dx)
    deck.ys = (0.0, 0.0, (ny - 0.5) * deck.dx, (ny - 0.5) * deck.dx)
    deck.xmax_domain = np.array([2.0 + nx * deck.dx, 2.0 + ny * deck.dx])
    sim = sps.Simulation.from_deck(deck)
    rng = np.random.default_rng(5)
    st = sps.initial_state(sim.parts, sim.niv)
    st.pop("x_10"), st.pop("disp_10")           # the outside approach's
    for k in ("vel", "stress", "f_drucker", "internal_vars"):
        st[k] = rng.standard_normal(st[k].shape)
    sim.set_state(st)
    for name, fields in SUBSETS.items():
        print(f"[read back] {nx} x {ny} {name}", flush=True)
        for _ in range(2):                      # the second from the buffers of the first
            out = sim.get_state(fields)
            for k in fields or st:
                assert bits_equal(out[k], st[k]), f"{name}: {k}"


# The staging on the device: at most 256 MiB for fields taken together (the
# state of this body has 450 MB), or the one field that is larger.
def test_staging_is_bounded():
    sps = load_pkg()
    lib = ctypes.CDLL(sps.PRODUCT_LIB)

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    nx = 1100
    deck = dataclasses.replace(sps.read_deck(deck_dir("t3_elastic")))
    deck.xs = (0.0, (nx - 0.5) * deck.dx, 0.0, (nx - 0.5) * deck.dx)
    deck.ys = (0.0, 0.0, (nx - 0.5) * deck.dx, (nx - 0.5) * deck.dx)
    deck.xmax_domain = np.array([2.0, 2.0]) + nx * deck.dx
    sim = sps.Simulation.from_deck(deck)
    st = sps.initial_state(sim.parts, sim.niv)
    small = sim.get_state(["f_drucker"])
    free = free_bytes()
    print(f"[read back] {sim.n2} particles, staging", flush=True)
    out = sim.get_state()
    taken = free - free_bytes()
    assert taken <= (256 << 20) + (4 << 20), f"{taken / 2**20:.0f} MiB"
    assert all(bits_equal(out[k], st[k]) for k in ("x", "vel", "stress", "internal_vars"))
    assert bits_equal(out["f_drucker"], small["f_drucker"])
