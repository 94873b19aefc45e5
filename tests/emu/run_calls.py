"""Sequences of calls on the CPU build of the HIP kernels (run under
AddressSanitizer by tests/test_emu_calls.py): `run_calls.py EMU_LIB NAME`.
Prints one line; exit status 0 when the sequence gives what it should."""
import ctypes
import dataclasses
import importlib
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path.insert(0, ROOT)
sps = importlib.import_module("stress-particle-sph_amd")
surrogate = importlib.import_module("stress-particle-sph_amd.surrogate")


def deck_of(name):
    return sps.read_deck(os.path.join(ROOT, "stress-particle-sph_amd", "decks", name))


def equal(a, b):
    return a.shape == b.shape and a.tobytes() == b.tobytes()


def same_state(a, b):
    a, b = a.get_state(), b.get_state()
    return [k for k in a if not equal(a[k], b[k])]


def direct_and_captured(lib, deck, parts=None):
    """The mixed form with kept lists, launched step by step and replayed."""
    sims = []
    for graph in (False, True):
        sim = sps.Simulation.from_deck(deck, lib_path=lib, mode=sps.MODE_FAST, parts=parts)
        sim.set_list_skin(0.25 * sim.params.dx)
        sim.set_graph(graph)
        sims.append(sim)
    return sims


def plastic_log_after_capture(lib):
    """A log set before and after a step was captured, made longer (another
    buffer) and taken away."""
    bad = []
    for caps in ((None, 16, 4096, 0), (16, 4096, 0)):
        sims = direct_and_captured(lib, deck_of("t2_cspm"))
        for k, cap in enumerate(caps):
            logs = []
            for sim in sims:
                if cap is not None:
                    surrogate.log_plastic(sim, cap)
                sim.step(4 if k else 12)     # the deck yields from its tenth step on
                logs.append(surrogate.plastic_log(sim, cap or 1))
            rows = [len(g[0]) for g in logs]
            if rows[0] != rows[1] or any(not equal(np.sort(a, axis=0), np.sort(b, axis=0)) for a, b in zip(*logs)):
                bad.append(f"log of {cap}: {rows[0]} rows, captured {rows[1]}")
            if cap and not rows[0]:
                bad.append(f"log of {cap} is empty")
        bad += same_state(*sims)
    return bad


def prescribed_values_after_capture(lib):
    """Other prescribed variables (the components exchanged) after a step was captured."""
    deck = deck_of("l1_localisation")
    sims = direct_and_captured(lib, deck)
    for sim in sims:
        sim.step(3)
    before = sims[0].get_state(["vel"])["vel"]
    other = dataclasses.replace(deck, bc_list=np.array(deck.bc_list))
    var = other.bc_list[:, 1]
    other.bc_list[:, 1] = np.select([var == 5, var == 6], [6, 5], var)
    if equal(other.bc_list, np.array(deck.bc_list)):
        return ["the deck prescribes no velocities"]
    for sim in sims:
        sim.set_bcs(other, sim.parts)
        sim.step(3)
    return same_state(*sims) + (["nothing moved"] if equal(before, sims[0].get_state(["vel"])["vel"]) else [])


def network_attached_again_after_capture(lib):
    """A network whose work buffers grow, when a larger simulation takes it
    too, after a step with it was captured."""
    net = surrogate.Network(ctypes.CDLL(lib), seed=3, batch_rows=64)
    sims = direct_and_captured(lib, deck_of("t2_cspm"))
    for sim in sims:
        surrogate.attach(sim, net, 1e4, 1e4)
        sim.step(12)     # the deck yields from its tenth step on
    if not surrogate.stats(sims[0])[0]:
        return ["the network was not used"]
    larger = sps.Simulation.from_deck(deck_of("v3_vslope_sp3"), lib_path=lib, mode=sps.MODE_FAST)
    surrogate.attach(larger, net, 1e4, 1e4)
    for sim in sims:
        sim.step(2)
    return same_state(*sims)


def block(nx):
    """An elastic block of nx x nx nodes."""
    deck = dataclasses.replace(deck_of("t3_elastic"))
    deck.xs = (0.0, (nx - 0.5) * deck.dx, 0.0, (nx - 0.5) * deck.dx)
    deck.ys = (0.0, 0.0, (nx - 0.5) * deck.dx, (nx - 0.5) * deck.dx)
    deck.xmax_domain = np.array([2.0, 2.0]) + nx * deck.dx
    return deck


def state_after_failed_event(lib):
    """The state taken back when an event of the read-back could not be
    created: an error, and the state from the next call."""
    sim = sps.Simulation.from_deck(block(250), lib_path=lib)   # a field takes more than one chunk
    want = sps.initial_state(sim.parts, sim.niv)
    emu = ctypes.CDLL(lib)
    emu.emu_set_events_left(1)
    bad = []
    try:
        sim.get_state(["x", "vel"])
        bad.append("no error")
    except sps.SpsError:
        pass
    emu.emu_set_events_left(-1)
    got = sim.get_state(["x", "vel"])
    return bad + [k for k in got if not equal(got[k], want[k])]


def state_short_of_memory(lib):
    """The state taken back where the device has room for its largest field
    and no more."""
    sim = sps.Simulation.from_deck(block(120), lib_path=lib)
    want = sps.initial_state(sim.parts, sim.niv)
    ctypes.CDLL(lib).emu_set_memory(32 * sim.n2 + 256)
    got = sim.get_state()
    return [k for k in ("x", "vel", "stress", "mass", "internal_vars", "x00") if not equal(got[k], want[k])]


def small_state_without_events(lib):
    """What fits one chunk is taken back with a copy and a wait, no event."""
    sim = sps.Simulation.from_deck(deck_of("t3_elastic"), lib_path=lib)
    want = sps.initial_state(sim.parts, sim.niv)
    ctypes.CDLL(lib).emu_set_events_left(0)
    got = sim.get_state()
    return [k for k in ("x", "vel", "stress", "mass", "internal_vars", "x00") if not equal(got[k], want[k])]


def lists_short_of_memory(lib):
    """Bodies whose lists of storage slots, and longer lists for several stress
    points a cell, do not fit beside the rest: the same steps without them."""
    emu = ctypes.CDLL(lib)
    emu.emu_memory_used.restype = ctypes.c_longlong
    bad = []
    for name, mode, least in (("t5_sp4", sps.MODE_ORDERED, 0.5), ("t4_xsph", sps.MODE_ORDERED, 0.9),
                              ("t3_elastic", sps.MODE_FAST, 0.9)):
        sims, used = [], []
        for limit in (None, least):
            before = emu.emu_memory_used()
            if limit:
                emu.emu_set_memory(int(limit * used[0]))
            deck = deck_of(name)
            parts = sps.build_particles(deck)
            sim = sps.Simulation(sps.make_params(deck, parts, mode=mode), lib)
            used.append(emu.emu_memory_used() - before)
            emu.emu_set_memory(-1)
            sim.set_state(sps.initial_state(parts, sim.niv))
            sim.deck, sim.parts = deck, parts
            sim.step(4)
            sims.append(sim)
        print(f"{name}: {used[0]} and {used[1]} bytes")
        bad += [f"{name}: {k}" for k in same_state(*sims)]
        for sim in sims:
            sim.close()
    return bad


def state_refused(lib):
    """A state that is refused leaves the one before, and its captured step;
    one that finds no memory leaves none to step on."""
    deck = deck_of("c1_collapse")
    deck.xs, deck.ys = (0.0, 5.5 * deck.dx, 0.0, 5.5 * deck.dx), (0.0, 0.0, 5.5 * deck.dx, 5.5 * deck.dx)
    sims = direct_and_captured(lib, deck)
    small = sps.initial_state(sims[0].parts, sims[0].niv)
    small["hsml"] = 0.3 * small["hsml"]       # less than the wall force's reach, and a larger grid
    bad = []

    def refused(what, call, code):
        try:
            call()
            bad.append(f"{what}: no error")
        except sps.SpsError as e:
            if e.code != code:
                bad.append(f"{what}: {e}")

    for sim in sims:
        sim.step(2)
    refused("small h", lambda: sims[1].set_state(small), -1)
    for sim in sims:
        sim.step(2)
    bad += same_state(*sims)
    small["hsml"] = 1.5 * small["hsml"]
    emu = ctypes.CDLL(lib)
    emu.emu_set_memory(0)
    refused("no memory", lambda: sims[1].set_state(small), -2)
    emu.emu_set_memory(-1)
    refused("step", lambda: sims[1].step(1), -5)
    sims[1].set_state(small)
    sims[1].step(1)
    return bad


def network_without_memory(lib):
    """A network that finds no memory to grow for a larger simulation: an
    error there, and in the next step of the one that used it; both work once
    it has grown."""
    net = surrogate.Network(sps.load_library(lib), seed=3, batch_rows=64)
    first = direct_and_captured(lib, deck_of("t2_cspm"))[1]
    surrogate.attach(first, net, 1e4, 1e4)
    first.step(12)
    larger = sps.Simulation.from_deck(deck_of("v3_vslope_sp3"), lib_path=lib, mode=sps.MODE_FAST)
    emu, bad = ctypes.CDLL(lib), []

    def refused(what, call):
        try:
            call()
            bad.append(f"{what}: no error")
        except sps.SpsError as e:
            if e.code != -2:
                bad.append(f"{what}: {e}")

    emu.emu_set_memory(1 << 20)
    refused("attach", lambda: surrogate.attach(larger, net, 1e4, 1e4))
    emu.emu_set_memory(-1)
    refused("step", lambda: first.step(1))
    refused("forward", lambda: net.forward(np.zeros((3, 10), dtype=np.float32)))
    larger.step(1)                               # without the network
    surrogate.attach(larger, net, 1e4, 1e4)
    larger.step(1)
    first.set_state(sps.initial_state(first.parts, first.niv))
    first.step(12)
    return bad


def materials_without_memory(lib):
    """A larger table of materials that finds no memory leaves the one before."""
    sims = direct_and_captured(lib, deck_of("t3_elastic"))
    p = sims[0].params
    row = [p.props[12], p.props[13], p.props[2], p.props[3], p.D11, p.D22, p.D12, p.D33, p.D41, p.D42]
    mat = np.zeros(sims[0].n2, dtype=np.int32)
    for sim in sims:
        sim.set_materials(np.array([row]), mat)
        sim.step(2)
    bad = []
    emu = ctypes.CDLL(lib)
    emu.emu_set_memory(0)
    try:
        sims[1].set_materials(np.array([row] * 50), mat)
        bad.append("no error")
    except sps.SpsError as e:
        if e.code != -2:
            bad.append(str(e))
    emu.emu_set_memory(-1)
    for sim in sims:
        sim.step(2)
    return bad + same_state(*sims)


CASES = {f.__name__: f for f in (plastic_log_after_capture, prescribed_values_after_capture,
                                 network_attached_again_after_capture, state_after_failed_event,
                                 state_short_of_memory, small_state_without_events,
                                 lists_short_of_memory, state_refused,
                                 network_without_memory, materials_without_memory)}

if __name__ == "__main__":
    bad = CASES[sys.argv[2]](sys.argv[1])
    print(f"{sys.argv[2]}: " + ("ok" if not bad else "; ".join(bad)))
    sys.exit(1 if bad else 0)
