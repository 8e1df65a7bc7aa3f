"""The super-steps' vector sums round as they are written down.

Assembled operators: the adjoint of a super-step is one fused multiply-add per
term, in the order the terms come in (mu L_j and mu_hat A^T L_j onto what stage
j + 1 left, nu, 1 - mu - nu and gamma_hat onto L_0's sum), computed here exactly
and rounded after each term from the transposed operator's own bits.  Operators
that read grad T: the stages in one call give the bits of the same stages as
vector operations (a time step per particle takes those), forward, and for
flux-limited diffusion backward.
"""
from fractions import Fraction

import numpy as np
import pytest

from sph_playground_amd import consts as C
from sph_playground_amd import problems as P

pytestmark = pytest.mark.gpu


def fma(a, b, c):
    return np.array([float(Fraction(float(x)) * Fraction(float(y)) + Fraction(float(z)))
                     for x, y, z in zip(np.broadcast_to(a, b.shape), b, np.broadcast_to(c, b.shape))])


@pytest.mark.parametrize("s", [2, 3, 5])
def test_adjoint_super_step_is_its_terms_in_order(gpu, s):
    import torch
    from sph_playground_amd import autograd as AG
    from sph_playground_amd.engine import Engine, sts_coeffs
    state, st = P.diffusion2d(12, b=(1.0, 0.3, 0.0), disotropic="no", seed=4, jitter=0.05)
    n, dt, K = st.shape[0], 1e-3, np.array([1.0, 0.4, 0.1, 0.2, 0.0, 0.0])
    rng = np.random.default_rng(3)
    T0, g = (torch.from_numpy(rng.standard_normal(n)).cuda() for _ in range(2))
    eng = Engine(state, kernel="m6", tensor="full", kappa_perp=0.1)
    eng.load(st)
    AG.prepare(eng)
    T0.requires_grad_(True)
    AG.sts(T0, torch.from_numpy(K), eng, s, dt, 1).backward(g)

    def transposed(lam):
        lam = torch.from_numpy(lam).cuda()
        return AG.apply_adjoint(eng, K, lam, lam, None)[0].cpu().numpy()

    lam, above, nu_above, base = g.cpu().numpy(), None, 0.0, np.zeros(n)
    for j in range(s, 1, -1):
        mu, nu, mh, gh = sts_coeffs(j, s)
        u = transposed(lam)
        low = fma(mh * dt, u, fma(mu, lam, nu_above * above if above is not None else np.zeros(n)))
        base = fma(gh * dt, u, fma(1.0 - mu - nu, lam, fma(nu, lam, base) if j == 2 else base))
        lam, above, nu_above = low, lam, nu
    want = fma(sts_coeffs(1, s)[2] * dt, transposed(lam), base + lam)
    assert np.array_equal(T0.grad.cpu().numpy(), want)
    eng.close()


def _fld():
    state, st = P.diffusion2d(12, seed=4, jitter=0.05)
    state[C.ec_eqs - 1] = C.eeq_manual
    state[C.ec_eqondiff - 1] = state[C.ec_eqonfluxlim - 1] = 1
    st[:, C.es_t - 1] += 2.0
    return state, st


@pytest.mark.parametrize("make,backward", [(lambda: P.diffusion2d(12, ddw="2nw-+", seed=4, jitter=0.05), False),
                                           (lambda: P.diffusion2d(12, ddw="2nw+-", seed=4, jitter=0.05), False),
                                           (_fld, True)], ids=["2nw-+", "2nw+-", "fld"])
def test_stages_in_one_call_are_the_vector_operations(gpu, make, backward):
    import torch
    from sph_playground_amd import autograd as AG
    from sph_playground_amd.engine import Engine
    state, st = make()
    n, dt = st.shape[0], 1e-5
    K = None if backward else torch.tensor([1.0, 0.4, 0.1, 0.2, 0.0, 0.0], dtype=torch.float64)
    eng = Engine(state, kernel="m6")
    eng.load(st)
    AG.prepare(eng)
    g = torch.from_numpy(np.random.default_rng(3).standard_normal(n)).cuda()
    outs = []
    for step in (dt, torch.full((n,), dt, dtype=torch.float64, device="cuda")):
        T0 = torch.from_numpy(st[:, C.es_t - 1].copy()).cuda().requires_grad_(backward)
        T = AG.sts(T0, K, eng, 4, step, 3, every=2)
        if backward:
            T.backward(g)
        outs.append((T.detach(), T0.grad))
    assert torch.equal(outs[0][0], outs[1][0])
    if backward:
        assert torch.equal(outs[0][1], outs[1][1])
    eng.close()
