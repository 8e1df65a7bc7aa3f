"""Leapfrog passes queued without a host round trip, against the oracle.

Between the passes the particles are ordered by counting them per cell (by the
sort where the last fullest cell held more than 256), the extended search grid
is filled into the room of the last one (and built again when it does not fit),
and the time step is reduced on the device.  Each pass is compared with the
oracle's iterate under the predictor and corrector of the reference's loop
(main.f90:241-362): the same neighbour sets, the time step within 1e-12, and
the fields within 1e-10 of each field's largest value (three steps, each moved
by its rounding, about 1e-15, times the few hundred terms of a sum and the
divergence of the predictor's positions).
"""
import numpy as np
import pytest

from oracle import oracle
from sph_playground_amd import consts as C
from sph_playground_amd import problems as P
from tests import goldens as G

pytestmark = pytest.mark.gpu

RATES = [("vx", "ax"), ("vy", "ay"), ("u", "du"), ("h", "dh"), ("t", "ddt")]


def _moving(side, seed=3, h_entry=1.0):
    state, st = P.hydro2d(side, seed=seed, jitter=0.05)
    st[:, C.es_vx - 1] = np.sin(np.pi * st[:, 1])
    st[:, C.es_vy - 1] = 0.5 * np.cos(2 * np.pi * st[:, 0])
    st[:, C.es_h - 1] *= h_entry
    return state, st


def _crowded():
    # a lattice of 24^2 and, within a cell or four of it, one of 36^2
    state, st = _moving(24)
    wide = st.shape[0]
    full = np.concatenate([st, st[np.arange(36 * 36) % wide]])
    k = np.arange(36 * 36)
    jit = 1e-5 * P.gaussian(11, 2 * k.size).reshape(-1, 2)
    full[wide:, 0] = 0.3 + 5e-4 * (k % 36) + jit[:, 0]
    full[wide:, 1] = 0.3 + 5e-4 * (k // 36) + jit[:, 1]
    full[wide:, C.es_h - 1] = 6e-4
    full[:, C.es_m - 1] = st[0, C.es_m - 1]
    full[wide:, C.es_m - 1] *= (5e-4 / (2.0 / 24)) ** 2
    state[C.ec_realpn - 1] = full.shape[0]
    return state, full


CASES = [("16", lambda: _moving(4), 1), ("256", lambda: _moving(16), 2), ("289", lambda: _moving(17), 2),
         # more particles than the time step's blocks hold threads
         ("66049", lambda: _moving(257), 2),
         ("walls", lambda: P.hydro2d_mti_walls(17, seed=4, jitter=0.05, velocity_seed=6), 2),
         ("crowded", _crowded, 2),
         # h grows on the first iterate, and the next grid's images with it
         ("grid_grows", lambda: _moving(12, h_entry=0.6), 2)]


def reference_passes(state, st, passes):
    """(store, dt, iterate's result) after every pass of the loop."""
    nr = int(state[C.ec_realpn - 1])
    col = lambda a, f: a[:, getattr(C, "es_" + f) - 1]
    out = oracle.iterate(state, st, kernel=1, neigh_cap=2000)
    for _ in range(passes):
        a = out["store"].copy()
        dt = 0.3 * col(a, "h")[:nr].min() / col(a, "c")[:nr].max()
        old = {k: col(a, k).copy() for _, k in RATES}
        for x, v, k in (("rx", "vx", "ax"), ("ry", "vy", "ay")):
            col(a, x)[:] = col(a, x) + dt * col(a, v) + 0.5 * dt * dt * old[k]
        for y, k in RATES:
            col(a, y)[:] = col(a, y) + dt * old[k]
        out = oracle.iterate(state, a, kernel=1, neigh_cap=2000)
        b = out["store"]
        for y, k in RATES:
            col(b, y)[:] = col(b, y) + 0.5 * dt * (col(b, k) - old[k])
        yield b, dt, out


@pytest.mark.parametrize("name,make,passes", CASES, ids=[c[0] for c in CASES])
def test_passes_match_oracle(gpu, name, make, passes):
    from sph_playground_amd.engine import Engine
    state, st = make()
    nr = int(state[C.ec_realpn - 1])
    eng = Engine(state, kernel="m6", neigh_cap=2000)
    eng.load(st)
    eng.step()
    records = [eng.stats()["ext_records"]]
    for b, dt, out in reference_passes(state, st, passes):
        print("case", name, flush=True)
        assert eng.leapfrog(1e30) == pytest.approx(dt, rel=1e-12)
        records.append(eng.stats()["ext_records"])
        off, j, code = eng.neighbours()
        assert G.pair_sets(out["off"], out["j"], out["code"]) == G.pair_sets(off, j, code)
        errs = G.field_errors(b, eng.save(), nr)
        assert max(errs.values()) <= 1e-10, errs
    if name == "grid_grows":  # past the room of the last grid, an eighth more than its records
        assert records[1] > records[0] + records[0] // 8
    eng.close()
