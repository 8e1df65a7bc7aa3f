"""Reverse neighbour lists of the prepared diffusion operator.

Short lists are filled through atomics and ordered per list, lists past 512
entries go through a sort of all pairs.  Both ways the transposed operator is
the transpose: <u, A v> = <A^T u, v> within 1e-12 of the sum of the terms'
sizes (n products, each rounded once: about 1e-16 sqrt(n) of it), and two
preparations of the same particles give the same bits.  M6 in 2D with uneven
radii: reverse lists longer and shorter than the forward ones; the Gaussian
kernel in 2D at hfac 1.4: some 615 neighbours.
"""
import numpy as np
import pytest

from sph_playground_amd import consts as C
from sph_playground_amd import problems as P

pytestmark = pytest.mark.gpu


def _uneven():
    # h at entry, which the lists are made with, varies by 25 %: not mutual
    state, st = P.diffusion2d(48, b=(1.0, 0.3, 0.0), disotropic="no", seed=4, jitter=0.05)
    st[:, C.es_h - 1] *= 1.0 + 0.25 * np.sin(2.0 * np.pi * st[:, 0])
    return state, st, "m6"


def _gauss():
    state, st = P.diffusion2d(60, hfac=1.4, b=(1.0, 0.3, 0.0), disotropic="no", kernel=C.KERNEL_GAUSS, seed=4,
                              jitter=0.05)
    return state, st, "gauss"


@pytest.mark.parametrize("make,longest", [(_uneven, (16, 512)), (_gauss, (513, 5000))], ids=["ordered", "sorted"])
def test_transpose_and_reproducibility(gpu, make, longest):
    import torch
    from sph_playground_amd import autograd as AG
    from sph_playground_amd.engine import Engine
    state, st, kernel = make()
    n = st.shape[0]
    K = np.array([1.0, 0.4, 0.1, 0.2, 0.0, 0.0])
    rng = np.random.default_rng(3)
    u, v = (torch.from_numpy(rng.standard_normal(n)).cuda() for _ in range(2))
    outs = []
    for _ in range(2):
        eng = Engine(state, kernel=kernel, tensor="full", kappa_perp=0.1)
        eng.load(st)
        AG.prepare(eng)
        off, j, _ = eng.neighbours()
        reverse = np.bincount(j, minlength=n).max()
        print(make.__name__, "longest reverse list", reverse, flush=True)
        assert longest[0] <= reverse <= longest[1]
        ATu, gA, _ = AG.apply_adjoint(eng, K, u, v, None)
        outs.append((AG.apply(eng, K, v), ATu, gA))
        eng.close()
    (Av, ATu, gA), (Av2, ATu2, gA2) = outs
    assert torch.equal(Av, Av2) and torch.equal(ATu, ATu2) and np.array_equal(gA, gA2)
    lhs, rhs = float(torch.dot(u, Av)), float(torch.dot(ATu, v))
    assert abs(lhs - rhs) <= 1e-12 * float(torch.dot(u.abs(), Av.abs())), (lhs, rhs)
