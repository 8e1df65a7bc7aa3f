"""Lanes per particle on each side of the lines that even lists draw, and every
field of the mixed path at each line.

Lattices whose lists are even at the first step (h at entry 1.03 spacings holds
whole shells of neighbours) lie on both sides of the sizes from which such lists
take one lane: FP64 within 1e-12 of each field's largest value (a vector's, over its
components: by symmetry some of them are rounding alone; a sum in another order
moves it by its rounding), the bar of the parity tests.

The mixed path is held to the FP64 oracle over the same three sweeps in which no
particle freezes (tolerance 1e-300), so that grad T and what reads it are taken
at the same h on both sides: every field loop 1 and loop 2 write, dT/dt, grad T
and the FLD velocity among them, within 1e-4 of the field's norm (a vector's, over
its components), the bar of the mixed-precision tests.

The FP32 sums of particles that move run in list order on one lane and on eight:
a step whose lists the step before found even gives the bits of a first step.
"""
import numpy as np
import pytest

from oracle import oracle
from sph_playground_amd import consts as C
from sph_playground_amd import problems as P
from tests.test_gpu_loop_lanes import CASES as LINES

pytestmark = pytest.mark.gpu

SCHEDULE = dict(max_sweeps=3, tol=1e-300)
FULL = dict(tensor="full", kappa_perp=0.1)
M4 = dict(kernel="m4")


def _diffusion(side, ddw, kernel=C.KERNEL_M6, hfac=1.0):
    return P.diffusion3d(side, ddw=ddw, b=(1.0, 0.4, 0.3), kind="square", h_scale=1.03, kernel=kernel, hfac=hfac)


def _varied(side):
    state, st = _diffusion(side, "fab")
    st[:, C.es_bx - 1] += 0.3 * np.sin(2.0 * np.pi * st[:, 1])
    return state, st


def _moving(side, equations="hydro", fld=False):
    n = side ** 3
    box = (0.0, 1.0, 0.0, 1.0, 0.0, 1.0)
    state, st = P.random_slab3d(n, box=box, hfac=1.0, equations=equations, fld=fld, lattice=(side,) * 3,
                                velocity_seed=2)
    pos, dx = P.lattice_positions(3, side, box)
    x = 2.0 * np.pi * pos[:, 0]
    st[:, 0:3] = pos
    for f, v in (("m", 1.0 / n), ("den", 1.0), ("h", 1.03 * dx), ("u", 1.5 + 0.3 * np.sin(x)), ("t", 1.0 + 0.2 * np.cos(x))):
        st[:, getattr(C, "es_" + f) - 1] = v
    P._eos_fill(st, 5.0 / 3.0)
    return state, st


EVEN = [
    # general form: from 110,000 particles in FP64, 150,000 in FP32
    ("2nw_47", lambda: _diffusion(47, "2nw-+"), FULL, ("fp64",)),
    ("2nw_48", lambda: _diffusion(48, "2nw-+"), FULL, ("fp64",)),
    ("2nw_sd_53", lambda: _diffusion(53, "2nw+-"), FULL, ("mixed",)),
    ("2nw_sd_54", lambda: _diffusion(54, "2nw+-"), FULL, ("mixed",)),
    # n2w and fw in FP32: from 225,000
    ("n2w_60", lambda: _diffusion(60, "n2w"), FULL, ("mixed",)),
    ("fw_61", lambda: _diffusion(61, "fw"), FULL, ("mixed",)),
    # fab with a B per particle in FP32: from 225,000
    ("fab_b_60", lambda: _varied(60), FULL, ("mixed",)),
    ("fab_b_61", lambda: _varied(61), FULL, ("mixed",)),
    # short lists (M4): moving in FP64 from 90,000 particles, 2nw from 75,000
    # and in FP32 from 120,000, fab in FP64 from 150,000 (hfac 1.2: 200,000)
    ("m4_hydro_44", lambda: _moving(44), M4, ("fp64",)),
    ("m4_hydro_45", lambda: _moving(45), M4, ("fp64",)),
    ("m4_2nw_42", lambda: _diffusion(42, "2nw-+", C.KERNEL_M4), dict(FULL, **M4), ("fp64",)),
    ("m4_2nw_43", lambda: _diffusion(43, "2nw-+", C.KERNEL_M4), dict(FULL, **M4), ("fp64",)),
    ("m4_2nw_sd_50", lambda: _diffusion(50, "2nw+-", C.KERNEL_M4), dict(FULL, **M4), ("mixed",)),
    ("m4_n2w_54", lambda: _diffusion(54, "n2w", C.KERNEL_M4), dict(FULL, **M4), ("fp64", "mixed")),
    ("m4_fab_59", lambda: _diffusion(59, "fab", C.KERNEL_M4, 1.2), dict(FULL, **M4), ("fp64", "mixed")),
]

VECTORS = (("ax", "ay", "az"), ("dbx", "dby", "dbz"), ("dtdx", "dtdy", "dtdz"))
SCALARS = ("den", "h", "om", "p", "c", "du", "dh", "ddt", "vfld")


def _check(state, st, precision, kw):
    from sph_playground_amd.engine import Engine
    nr = int(state[C.ec_realpn - 1])
    okw = {"neigh_cap": kw["neigh_cap"]} if "neigh_cap" in kw else {}
    if kw.get("tensor") == "full":
        okw.update(tensor_mode=1, kappa_perp=kw["kappa_perp"])
    if precision == "mixed" and state[C.ec_adden - 1] == C.YESNO["yes"]:
        okw.update(SCHEDULE)
        kw = dict(kw, max_sweeps=SCHEDULE["max_sweeps"], newton_tol=SCHEDULE["tol"])
    kw = dict({"kernel": "m6"}, **kw)
    ref = oracle.iterate(state, st, kernel=C.KERNELS[kw["kernel"]], **okw)
    eng = Engine(state, precision=precision, **kw)
    got = st.copy()
    eng.iterate(got)
    assert eng.stats()["n_pairs"] == ref["off"][-1] and eng.stats()["sweeps"] == ref["sweeps"]
    eng.close()
    ref = ref["store"]
    norms = {}
    for group in VECTORS + tuple((f,) for f in SCALARS):
        k = [getattr(C, "es_" + f) - 1 for f in group]
        diff = got[:nr, k] - ref[:nr, k]
        norms[group] = np.linalg.norm(ref[:nr, k])
        print(group, "%.1e of %.1e" % (np.linalg.norm(diff), norms[group]), flush=True)
        if precision == "fp64":
            assert np.abs(diff).max() <= 1e-12 * np.abs(ref[:nr, k]).max(), group
        else:
            assert np.linalg.norm(diff) <= 1e-4 * norms[group], group
    assert norms[VECTORS[0]] > 0.0 or norms[("ddt",)] > 0.0  # loop 2 wrote something


@pytest.mark.parametrize("name,make,kw,precision", [(n, m, kw, p) for n, m, kw, ps in EVEN for p in ps],
                         ids=["%s-%s" % (e[0], p) for e in EVEN for p in e[3]])
def test_even_lists_on_each_side(gpu, name, make, kw, precision):
    print("case", name, precision, flush=True)
    state, st = make()
    _check(state, st, precision, kw)


@pytest.mark.parametrize("name,make,kw", LINES, ids=[c[0] for c in LINES])
def test_every_field_of_the_mixed_path(gpu, name, make, kw):
    print("case", name, flush=True)
    state, st = make()
    _check(state, st, "mixed", kw)


def _simple1d(n):
    state, st = P.hydro1d(n)
    state[C.ec_adden - 1] = C.YESNO["no"]
    return state, st


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("make", [lambda: _simple1d(1000), lambda: P.hydro2d(199, seed=3, jitter=0.05, adden="no"),
                                  lambda: P.hydro2d(201, seed=3, jitter=0.05, adden="no"),
                                  lambda: P.hydro2d(388, seed=3, jitter=0.05, adden="no"),
                                  lambda: P.diffusion3d(34, ddw="2nw+-", adden="no", kind="square", h_scale=1.03),
                                  lambda: P.diffusion3d(35, ddw="2nw+-", adden="no", kind="square", h_scale=1.03)],
                         ids=["1d", "2d_199", "2d_201", "2d_388", "3d_34", "3d_35"])
def test_direct_summation_on_each_side(gpu, make, precision):
    # c1simple takes loop 1's lanes of uneven lists in FP64, one in FP32
    state, st = make()
    _check(state, st, precision, {})


@pytest.mark.parametrize("kernel", ["m4", "m6"])
@pytest.mark.parametrize("equations,fld", [("hydro", False), ("magnetohydro", False), ("hydro", True), ("hydi", False)],
                         ids=["hydro", "mhd", "fld", "hydi"])
def test_even_lists_of_moving_particles_keep_their_bits(gpu, equations, fld, kernel):
    # 56^3 = 175,616 particles; cells of a quarter radius hold one particle
    # each, so their order is the same however it came about
    from sph_playground_amd.engine import Engine
    state, st = _moving(56, equations, fld)
    eng = Engine(state, kernel=kernel, precision="mixed", cell_div=4)
    eng.load(st)
    eng.step()
    first = eng.save()
    eng.step()
    second = eng.save()
    eng.load(first)
    eng.step()
    assert np.array_equal(eng.save(), second)
    eng.close()
