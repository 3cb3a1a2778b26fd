"""clip_grad_norm on both sides of the size up to which its scaling launch keeps the gradients in the cache."""
import pytest
import torch

from tests.util import assert_parity

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("extra", [-5, 0, 5])
def test_gradients_around_the_cached_size(dtype, extra):
    from cubework_amd.clip_grad import clip_grad_norm

    n = (64 << 20) // dtype.itemsize + extra
    params = []
    for k, size in enumerate((n // 2 + 3, n - n // 2 - 3)):
        p = torch.nn.Parameter(torch.empty(size, dtype=dtype, device=DEV))
        p.grad = torch.randn(size, dtype=dtype, device=DEV, generator=torch.Generator(device=DEV).manual_seed(k)) * 0.01
        params.append(p)
    before = [p.grad.double() for p in params]
    norm = clip_grad_norm(params, 1.0)
    want = torch.sqrt(sum((g * g).sum() for g in before))
    assert_parity(norm, want.cpu(), torch.float32, "norm of %d elements" % n)
    for p, g in zip(params, before):
        assert_parity(p.grad, (g / want).cpu(), dtype, "clipped gradient of %d elements" % n)
