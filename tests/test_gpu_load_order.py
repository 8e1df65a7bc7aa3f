"""Loading orders the particles by search cell; what is loaded stays the caller's.

A store's rows come back in the caller's order, bit for bit, whatever their
order, also where they cannot be ordered (a coordinate or h that is no finite
number); the first step on shuffled rows is the oracle's (fields within 1e-12 of
each field's largest value, the bar of the parity tests, and the same
neighbour sets), also where particles left the box and are wrapped, and a
second load replaces the first.  Sizes at the edges of the transposition's
tiles of 64 rows.
"""
import numpy as np
import pytest

from oracle import oracle
from sph_playground_amd import consts as C
from sph_playground_amd import problems as P
from tests import goldens as G

pytestmark = pytest.mark.gpu


def _shuffled(side, seed, walls=False):
    state, st = (P.hydro2d_mti_walls if walls else P.hydro2d)(side, seed=seed, jitter=0.05)
    nr = int(state[C.ec_realpn - 1])
    order = np.concatenate([np.random.default_rng(seed).permutation(nr), np.arange(nr, st.shape[0])])
    return state, np.ascontiguousarray(st[order])


@pytest.mark.parametrize("escaped", [0, 3], ids=["inside", "escaped"])
@pytest.mark.parametrize("side,walls", [(4, False), (8, False), (9, False), (23, False), (17, True)])
def test_first_step_of_shuffled_rows_matches_oracle(gpu, side, walls, escaped):
    from sph_playground_amd.engine import Engine
    state, st = _shuffled(side, 5, walls)
    nr = int(state[C.ec_realpn - 1])
    st[:escaped, 0] = 2.0 * np.sign(st[:escaped, 0]) - st[:escaped, 0]  # as far outside the box as it was inside
    eng = Engine(state, kernel="m6")
    eng.load(np.ascontiguousarray(st[::-1][:nr]))  # replaced by the next load
    eng.load(st)
    assert np.array_equal(eng.save(), st)
    eng.step()
    ref = oracle.iterate(state, st, kernel=1)
    off, j, code = eng.neighbours()
    assert G.pair_sets(ref["off"], ref["j"], ref["code"]) == G.pair_sets(off, j, code)
    errs = G.field_errors(ref["store"], eng.save(), nr)
    assert max(errs.values()) <= 1e-12, errs
    eng.close()


@pytest.mark.parametrize("column,value", [("rz", np.inf), ("rx", np.nan), ("h", np.inf), ("h", 0.0), ("h", -1.0)])
def test_rows_that_cannot_be_ordered_come_back(gpu, column, value):
    from sph_playground_amd.engine import Engine
    state, st = _shuffled(9, 6)
    st[:, getattr(C, "es_" + column) - 1] = value
    eng = Engine(state, kernel="m6")
    eng.load(st)
    assert np.array_equal(eng.save(), st, equal_nan=True)
    eng.close()
