"""Reverse lists longer than the room they are first given, and room kept from
another store.

60 particles on a ring reach the one at its centre, which reaches none: its
reverse list is 60 long where the longest forward one is 21 and the first room
24, so the lists are filled a second time.  The transposed operator is then the
transpose of the dense matrix that single columns give, within 1e-13 of its
largest entry (each entry is one pair's weight, or a row's sum of 21).  A
preparation that finds the buffers of a store with longer, or shorter, lists
gives the bits of one on a fresh context.
"""
import numpy as np
import pytest

from sph_playground_amd import consts as C
from sph_playground_amd import problems as P

pytestmark = pytest.mark.gpu

K = np.array([1.0, 0.4, 0.1, 0.2, 0.0, 0.0])


def _ring(ddw, m=60, radius=0.12):
    state, few = P.diffusion2d(8, ddw=ddw, b=(1.0, 0.3, 0.0), disotropic="no", hfac=1.4, adden="no")
    st = np.repeat(few[:1], m + 1, 0)
    angle = 2.0 * np.pi * np.arange(m) / m
    st[:, 0:2] = 0.5
    st[:m, 0] += radius * np.cos(angle)
    st[:m, 1] += radius * np.sin(angle)
    st[:, C.es_m - 1] = 1.0 / m
    st[:m, C.es_h - 1] = 1.02 * radius / 3.0
    st[m, C.es_h - 1] = radius / 10.0
    state[C.ec_realpn - 1] = m + 1
    return state, st


@pytest.mark.parametrize("ddw", ["fab", "n2w", "2nw-+"])
def test_lists_past_the_room(gpu, ddw):
    import torch
    from sph_playground_amd import autograd as AG
    from sph_playground_amd.engine import Engine
    state, st = _ring(ddw)
    n = st.shape[0]
    eng = Engine(state, kernel="m6", tensor="full", kappa_perp=0.1)
    eng.load(st)
    AG.prepare(eng)
    off, j, _ = eng.neighbours()
    assert np.diff(off).max() == 21 and np.bincount(j, minlength=n).max() == 60
    eye = torch.eye(n, dtype=torch.float64, device="cuda")
    A = torch.stack([AG.apply(eng, K, e) for e in eye], 1)
    AT = torch.stack([AG.apply_adjoint(eng, K, e, e, None)[0] for e in eye], 1)
    assert A[:, -1].abs().max() > 0.0  # the centre enters the ring's rows
    assert (AT - A.T).abs().max() <= 1e-13 * A.abs().max()
    eng.close()


def test_room_of_another_store(gpu):
    import torch
    from sph_playground_amd import autograd as AG
    from sph_playground_amd.engine import Engine
    state, wide = P.diffusion2d(24, b=(1.0, 0.3, 0.0), disotropic="no", seed=4, jitter=0.05, adden="no")
    narrow = wide.copy()
    narrow[:, C.es_h - 1] *= 0.7
    v = torch.from_numpy(np.random.default_rng(3).standard_normal(wide.shape[0])).cuda()

    def gradients(eng, st):
        eng.load(st)
        AG.prepare(eng)
        T0 = v.clone().requires_grad_(True)
        Kt = torch.from_numpy(K).requires_grad_(True)
        T = AG.sts(T0, Kt, eng, 3, 1e-4, 4, every=2)
        T.backward(v)
        return [AG.apply_adjoint(eng, K, v, v, None)[0], T.detach(), T0.grad, Kt.grad]

    used = Engine(state, kernel="m6", tensor="full", kappa_perp=0.1)
    for st in (wide, narrow, wide):
        fresh = Engine(state, kernel="m6", tensor="full", kappa_perp=0.1)
        for a, b in zip(gradients(used, st), gradients(fresh, st)):
            assert torch.equal(a, b)
        fresh.close()
    used.close()
