"""The pair loops at the sizes where the number of lanes per particle changes.

A step gives a particle 8, 4 or 1 lanes of loop 1 and loop 2 by the particle
count, the dimension, the equation set and (large diffusion sets) how even the
last lists were.  Lists of every length modulo 8 are split over the lanes, so
each side of each line is held to the oracle on jittered particles: FP64
within 1e-12 of each field's largest value (a sum over the list in another
order moves it by its rounding, about 1e-15), FP32 pair arithmetic with h, rho
and Omega within 1e-5 pointwise and the force fields within 1e-4 normwise, the
bars of the parity and mixed-precision tests.  The FP32 sums of loop 1, and of
loop 2 for particles that move, run in list order on one lane and on eight
alike.
"""
import numpy as np
import pytest

from oracle import oracle
from sph_playground_amd import consts as C
from sph_playground_amd import problems as P
from tests import goldens as G

pytestmark = pytest.mark.gpu


def _jitter(st, dim, amount, seed):
    n = st.shape[0]
    dx = (1.0 / n) ** (1.0 / dim)
    st[:, :dim] = (st[:, :dim] + amount * dx * P.gaussian(seed, dim * n).reshape(n, dim)) % 1.0
    return st


def _diffusion(side, ddw, jitter):
    state, st = P.diffusion3d(side, ddw=ddw, b=(1.0, 0.4, 0.3), kind="square")
    return state, _jitter(st, 3, jitter, 5) if jitter else st


CASES = [
    # 2D: 8 lanes below 40,000 particles, 4 below 150,000, then 1
    ("hydro2d_199", lambda: P.hydro2d(199, seed=3, jitter=0.05), {}),
    ("hydro2d_201", lambda: P.hydro2d(201, seed=3, jitter=0.05), {}),
    ("hydro2d_387", lambda: P.hydro2d(387, seed=3, jitter=0.05), {}),
    ("hydro2d_388", lambda: P.hydro2d(388, seed=3, jitter=0.05), {}),
    # 3D diffusion: 8 lanes below 40,000 particles, then 4 (2nw: 1 in loop 2
    # from 300,000 on); FP32 in loop 1 8 below 100,000, then 1
    ("fab_34", lambda: _diffusion(34, "fab", 0.05), dict(tensor="full", kappa_perp=0.1)),
    ("fab_35", lambda: _diffusion(35, "fab", 0.05), dict(tensor="full", kappa_perp=0.1)),
    ("fab_46", lambda: _diffusion(46, "fab", 0.05), dict(tensor="full", kappa_perp=0.1)),
    ("fab_47", lambda: _diffusion(47, "fab", 0.05), dict(tensor="full", kappa_perp=0.1)),
    ("n2w_35", lambda: _diffusion(35, "n2w", 0.05), dict(tensor="full", kappa_perp=0.1)),
    ("2nw_sd_35", lambda: _diffusion(35, "2nw+-", 0.05), dict(tensor="full", kappa_perp=0.1)),
    ("2nw_ds_67", lambda: _diffusion(67, "2nw-+", 0.05), dict(tensor="full", kappa_perp=0.1)),
    # particles that move in 3D: 8 lanes at every size
    ("mhd_50000", lambda: P.shock_slab_walls(50000, seed=5, hfac=1.2, equations="magnetohydro", velocity_seed=2),
     dict(neigh_cap=600)),
    ("hydro3d_5000", lambda: P.shock_slab_walls(5000, seed=6, hfac=1.2, velocity_seed=2), dict(neigh_cap=600)),
    ("fld_5000", lambda: P.shock_slab_walls(5000, seed=6, hfac=1.2, fld=True, velocity_seed=2), dict(neigh_cap=600)),
    # c1simple
    ("simple_35", lambda: P.diffusion3d(35, ddw="2nw-+", adden="no", kind="square"), {}),
]


def _compare(got, ref, nr, precision):
    if precision == "fp64":
        errs = G.field_errors(ref, got, nr)
        assert max(errs.values()) <= 1e-12, errs
        return
    for f in ("den", "h", "om"):
        k = getattr(C, "es_" + f) - 1
        assert (np.abs(got[:nr, k] - ref[:nr, k]) / np.abs(ref[:nr, k])).max() <= 1e-5, f
    for f in ("ax", "ay", "az", "du", "dbx", "dby", "dbz"):
        k = getattr(C, "es_" + f) - 1
        norm = np.linalg.norm(ref[:nr, k])
        assert np.linalg.norm(got[:nr, k] - ref[:nr, k]) <= 1e-4 * norm, f


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name,make,kw", CASES, ids=[c[0] for c in CASES])
def test_step_matches_oracle_on_each_side_of_the_lines(gpu, name, make, kw, precision):
    from sph_playground_amd.engine import Engine
    print("case", name, precision, flush=True)
    state, st = make()
    nr = int(state[C.ec_realpn - 1])
    okw = {"neigh_cap": kw["neigh_cap"]} if "neigh_cap" in kw else {}
    if kw.get("tensor") == "full":
        okw.update(tensor_mode=1, kappa_perp=kw["kappa_perp"])
    ref = oracle.iterate(state, st, kernel=1, **okw)
    eng = Engine(state, kernel="m6", precision=precision, **kw)
    got = st.copy()
    eng.iterate(got)
    assert eng.stats()["n_pairs"] == ref["off"][-1]
    _compare(got, ref["store"], nr, precision)
    eng.close()


def test_second_step_of_even_lists_matches_oracle(gpu):
    # 90^3 = 729,000 lattice particles: the first step has no lists to judge
    # by (4 lanes), the second finds them even (1 lane)
    from sph_playground_amd.engine import Engine
    state, st = P.diffusion3d(90, ddw="fab", b=(1.0, 1.0, 0.0))
    nr = st.shape[0]
    eng = Engine(state, kernel="m6", tensor="full", kappa_perp=1e-3)
    eng.load(st)
    eng.step()
    first = eng.save()
    eng.step()
    second = eng.save()
    for inp, out in ((st, first), (first, second)):
        ref = oracle.iterate(state, inp, kernel=1, tensor_mode=1, kappa_perp=1e-3)
        _compare(out, ref["store"], nr, "fp64")
    eng.close()
