"""Infinities in the mixed loop 2 stay infinities.

Particles so light that rho^2 leaves FP32 divide by zero: sums all of whose terms
have one sign are infinite, others NaN.  The sums of a fixed equation set, run in
list order on eight lanes over batches that lists do not fill, end as those of the
general kernel on one lane.  An expanding flow gives du/dt's terms one sign away
from the box's faces, where images jump; rho about 1e-22, u 1e22.
"""
import os

import numpy as np
import pytest

from sph_playground_amd import consts as C
from sph_playground_amd import problems as P

pytestmark = pytest.mark.gpu


def _step(state, st, generic):
    from sph_playground_amd.engine import Engine
    old = os.environ.pop("SPH_LOOP2_GENERIC", None)
    try:
        if generic:
            os.environ["SPH_LOOP2_GENERIC"] = "1"
        eng = Engine(state, kernel="m6", precision="mixed")
    finally:
        os.environ.pop("SPH_LOOP2_GENERIC", None)
        if old is not None:
            os.environ["SPH_LOOP2_GENERIC"] = old
    out = st.copy()
    eng.iterate(out)
    eng.close()
    return out


@pytest.mark.parametrize("equations,fld", [("hydro", False), ("magnetohydro", False), ("hydro", True)],
                         ids=["hydro", "mhd", "fld"])
def test_infinite_sums(gpu, equations, fld):
    state, st = P.random_slab3d(14 ** 3, seed=5, box=(0.0, 1.0, 0.0, 1.0, 0.0, 1.0), hfac=1.0, equations=equations,
                                fld=fld, artts="no", lattice=(14, 14, 14))
    st[:, C.es_m - 1] *= 1e-22
    st[:, C.es_den - 1] *= 1e-22
    st[:, C.es_u - 1] *= 1e22
    st[:, C.es_vx - 1:C.es_vz] = st[:, 0:3] - 0.5
    one, eight = _step(state, st, True), _step(state, st, False)
    inf = np.isinf(one[:, C.es_du - 1]).sum()
    print(equations, fld, "infinite du/dt", inf, flush=True)
    assert inf > 100
    for f in ("ax", "ay", "az", "du", "ddt", "dbx", "dby", "dbz"):
        k = getattr(C, "es_" + f) - 1
        assert np.array_equal(np.isnan(one[:, k]), np.isnan(eight[:, k])), f
        assert np.array_equal(np.isinf(one[:, k]), np.isinf(eight[:, k])), f
