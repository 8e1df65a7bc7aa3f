"""Super-steps of the grad T operators with an `every` that is no integer.

A forward run takes any number to space its checkpoints by; its stages one by one
give the bits of the same stages in one call.
"""
import pytest

from sph_playground_amd import consts as C
from tests.test_gpu_adjoint_nl import _K, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [2.0, 1.5, float("inf")])
def test_forward_takes_any_spacing(gpu, every):
    import torch
    state, st, eng, AG = _setup("2nw-+")
    T0 = torch.from_numpy(st[:, C.es_t - 1].copy()).cuda()
    K = torch.tensor(_K())
    assert torch.equal(AG.sts(T0, K, eng, 3, 2e-5, 4, every), AG.sts(T0, K, eng, 3, 2e-5, 4, 2))
    eng.close()
