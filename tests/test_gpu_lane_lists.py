"""A step's bits depend on the particles it starts from, not on earlier ones.

Large 3D diffusion sets take one lane per particle where the neighbour lists
are even and several where they are not, which rounds the sums otherwise; the
lists that count are the step's own.  90^3 = 729,000 particles, past the line:
the same store gives the same bits on a fresh engine, again on that engine and
after a store of uneven lists; and a step that was queued for lists like the
last step's, which were even, but finds its own uneven (h at entry 1.03 spacings
holds whole shells of the lattice within the radius, the solved h cuts one)
gives the bits of a first step on the same state.  Cells of a quarter radius hold
one particle each there, so their order is the same however it came about.
"""
import numpy as np
import pytest

from sph_playground_amd import consts as C
from sph_playground_amd import problems as P

pytestmark = pytest.mark.gpu

KW = dict(tensor="full", kappa_perp=1e-3, cell_div=4)


def _lattice(jitter, h_scale=1.0, side=90):
    state, st = P.diffusion3d(side, ddw="fab", b=(1.0, 1.0, 0.0), kind="square", h_scale=h_scale)
    if jitter:
        st[:, :3] = (st[:, :3] + jitter / side * P.gaussian(5, 3 * side ** 3).reshape(-1, 3)) % 1.0
    return state, st


def _lists(store, state, side):
    from oracle import oracle
    counts = np.diff(oracle.iterate(state, store, kernel=1, tensor_mode=1, kappa_perp=1e-3)["off"])
    return counts.max() / counts.mean()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_same_store_same_bits(gpu, precision):
    from sph_playground_amd.engine import Engine
    state, even = _lattice(0.0, 1.03)
    _, uneven = _lattice(0.05)
    eng = Engine(state, kernel="m6", precision=precision, **KW)
    outs = []
    for st in (even, even, uneven, even, uneven):
        print(precision, "store", len(outs), flush=True)
        eng.load(st)
        eng.step()
        outs.append(eng.save())
    eng.close()
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[3])
    assert np.array_equal(outs[2], outs[4])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lists_that_turn_uneven(gpu, precision):
    from sph_playground_amd.engine import Engine
    small_state, small = _lattice(0.01, 1.03, 18)  # the lists' shape does not depend on the size
    from oracle import oracle
    after = oracle.iterate(small_state, small, kernel=1, tensor_mode=1, kappa_perp=1e-3)["store"]
    assert _lists(small, small_state, 18) <= 1.05 < _lists(after, small_state, 18)
    state, st = _lattice(0.01, 1.03)
    eng = Engine(state, kernel="m6", precision=precision, **KW)
    eng.load(st)
    eng.step()
    first = eng.save()
    eng.step()
    second = eng.save()
    eng.close()
    eng = Engine(state, kernel="m6", precision=precision, **KW)
    eng.load(first)
    eng.step()
    assert np.array_equal(eng.save(), second)
    eng.close()
