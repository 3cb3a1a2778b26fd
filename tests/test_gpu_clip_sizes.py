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


@pytest.mark.parametrize("norm_type", [2.0, 1.0, 3.0, float("inf")])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 4095, 4097, 16384 + 1, 65536 - 8, 65536 + 8, (32 << 20) + 40, (64 << 20) + 40])
def test_norm_around_the_batches_of_loads(n, dtype, norm_type):
    """One tensor of sizes around a thread's vectors, a block's batches and chunk, and a launch's 128 MB."""
    from cubework_amd.clip_grad import clip_grad_norm

    p = torch.nn.Parameter(torch.empty(n, dtype=dtype, device=DEV))
    p.grad = torch.randn(n, dtype=dtype, device=DEV, generator=torch.Generator(device=DEV).manual_seed(n)) * 0.25
    want = torch.linalg.vector_norm(p.grad, norm_type, dtype=torch.float64)
    assert_parity(clip_grad_norm([p], 1e9, norm_type), want.cpu(), torch.float32, "norm %g of %d elements" % (norm_type, n))
