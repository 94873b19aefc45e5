"""The state taken back from the device, against the arrays it was set from,
bit for bit: fields that fit one staging chunk (1 MiB), that end in the
middle of one, and that take several per thread; every field at once, some,
one, and none."""
import ctypes
import dataclasses

import numpy as np
import pytest

from conftest import ORACLE_LIB, bits_equal, deck_dir, load_pkg

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


def poisoned(sps, sim, names):
    """The named fields, taken back into arrays full of a pattern."""
    out, st = {}, sps.State()
    for name in names:
        dt, shape = sim._shape(name)
        out[name] = np.frombuffer(b"\xa5" * (int(np.prod(shape)) * np.dtype(dt).itemsize), dtype=dt).reshape(shape).copy()
        setattr(st, name, out[name].ctypes.data)
    sim._check(sim.lib.sps_get_state(sim.handle, ctypes.byref(st)))
    return out


# After steps, when the storage is in the order of the cells: every field
# against the oracle's, with a value of its own at every particle, taken back
# together (several chunks, several threads) and one by one (other chunks).
# The outside approach adds x_10 and disp_10 and the surface, by original index.
@pytest.mark.parametrize("name,nx,ny", [("c1_collapse", 230, 190), ("c1_collapse", 23, 19), ("b4_bui_outside", 0, 0)])
def test_state_in_original_order(name, nx, ny):
    sps = load_pkg()
    deck = dataclasses.replace(sps.read_deck(deck_dir(name)))
    if nx:
        deck.xs = (0.0, (nx - 0.5) * deck.dx, 0.0, (nx - 0.5) * deck.dx)
        deck.ys = (0.0, 0.0, (ny - 0.5) * deck.dx, (ny - 0.5) * deck.dx)
        deck.dy = deck.dx
    parts = sps.build_particles(deck)
    gpu = sps.Simulation.from_deck(deck, parts=parts)
    ora = sps.Simulation.from_deck(deck, lib_path=ORACLE_LIB, parts=parts)
    print(f"[read back] {name}: {gpu.n2} particles in the order of the cells", flush=True)
    rng = np.random.default_rng(9)
    st = sps.initial_state(parts, gpu.niv)
    for k in ("x00", "displ", "f_drucker", "internal_vars"):
        st[k] = 1e-3 * rng.standard_normal(st[k].shape)
    for k in ("mass", "rho"):
        st[k] = st[k] * (1.0 + 1e-3 * rng.standard_normal(st[k].shape))
    st["vel"][:gpu.n] = 0.5 * rng.standard_normal((gpu.n, 2))
    st["if_out_domain"][rng.permutation(gpu.n2)[:gpu.n2 // 50]] = 1
    if not nx:
        st["disp_10"] = 1e-6 * rng.standard_normal(gpu.nn)
    else:
        st.pop("x_10"), st.pop("disp_10")
    for sim in (gpu, ora):
        sim.set_state(st)
        sim.step(3)
    names = [k for k in sps.State.__dict__ if k in st] + ["grad_u", "ddev_strn", "f_bound", "art_visc"]
    want = poisoned(sps, ora, names)
    got = poisoned(sps, gpu, names)
    bad = [k for k in names if not bits_equal(got[k], want[k])]
    bad += [f"{k} alone" for k in names if not bits_equal(poisoned(sps, gpu, [k])[k], want[k])]
    assert not bad, ", ".join(bad)
    flat = [k for k in ("x", "x00", "internal_vars", "f_drucker", "mass") if np.unique(got[k]).size < got[k].size / 2]
    assert not flat, f"many equal values: {flat}"
    if deck.update_x:
        for what, a, b in zip(("bc_or_not", "normal"), ora.get_surface(), gpu.get_surface()):
            assert bits_equal(a, b), what
