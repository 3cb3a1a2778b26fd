"""Casts of several tensors in one launch against torch's, bit for bit, and what a block under autocast does with them."""
import ctypes

import pytest
import torch

from tests.util import randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.bfloat16: 0, torch.float32: 1, torch.float16: 2}


def _cast(srcs, dtype):
    from cubework_amd import _lib
    dsts = [torch.full((s.numel() + 16,), float("nan"), dtype=dtype, device=DEV) for s in srcs]
    table = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])  # noqa: E731
    n = (ctypes.c_int64 * len(srcs))(*[s.numel() for s in srcs])
    rc = _lib.load().cw_cast_many(len(srcs), table(srcs), table(dsts), ctypes.cast(n, ctypes.c_void_p), CODE[srcs[0].dtype], CODE[dtype],
                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return rc, dsts


@pytest.mark.parametrize("src,dst", [(torch.float32, torch.float16), (torch.float32, torch.bfloat16), (torch.float16, torch.float32),
                                     (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("sizes", [(1,), (3, 4, 5, 7), (4095, 4096, 4097), (1024, 0, 12289, 2), (1 << 20, 1025)])
def test_casts_of_several_tensors(src, dst, sizes):
    srcs = [randn((n,), torch.float32, n + 1, std=100.0).to(src).to(DEV) for n in sizes]
    if src == torch.float32:  # overflow, subnormals of either type, ties, signed zeros
        special = torch.tensor([1e6, -1e38, 65520.0, 65519.9, 6e-8, 2.9e-8, 1e-40, -0.0, float("inf"), 1.00048828125, 1.00390625], device=DEV)
        srcs[-1][:special.numel()] = special[:srcs[-1].numel()]
    rc, got = _cast(srcs, dst)
    assert rc == 0
    for s, g in zip(srcs, got):
        assert torch.equal(g[:s.numel()], s.to(dst)) and torch.isnan(g[s.numel():]).all()


def test_refusals():
    x = randn((64,), torch.float32, 1, device=DEV)
    assert _cast([x[1:]], torch.float16)[0] == -2  # not 16-byte aligned
    assert _cast([x.half()], torch.bfloat16)[0] == -3
    assert _cast([x] * 5, torch.float16)[0] == -1


@pytest.mark.parametrize("amp", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_under_autocast_keeps_its_types(amp, dtype):
    """A block's parameters and stream in either type: the residual branch carries the input's own type, gradients the parameters'."""
    from cubework_amd.distributed import initialize
    from cubework_amd.opt_block import OPTBlock
    initialize("2d", 1)
    blk = OPTBlock(hidden=128, heads=2, ffn=512, dtype=dtype).to(DEV)
    g = torch.Generator(device=DEV).manual_seed(3)
    with torch.no_grad():
        for name, p in blk.named_parameters():
            p.copy_(torch.randn(p.shape, generator=g, device=DEV) * 0.05 + (1.0 if "norm" in name and name.endswith("weight") else 0.0))

    def run(plain):
        x = randn((2, 33, 128), dtype, 5, device=DEV).requires_grad_(True)
        keep = OPTBlock._norm_fork
        if plain:  # the two branches' gradients added by autograd
            OPTBlock._norm_fork = staticmethod(lambda layer, t: (layer(t), t))
        try:
            for p in blk.parameters():
                p.grad = None
            with torch.autocast("cuda", dtype=amp):
                y = blk(x)
            y.backward(torch.ones_like(y))
        finally:
            OPTBlock._norm_fork = staticmethod(keep)
        assert x.grad.dtype == dtype and all(p.grad.dtype == dtype for p in blk.parameters())
        return y, [x.grad] + [p.grad for p in blk.parameters()]

    y, grads = run(False)
    want, want_grads = run(True)
    assert y.dtype == want.dtype and torch.equal(y, want)
    # one fp32 addition in another place: what it changes is rounded to 16 bits on the way back
    bar = 2.0 ** (-9 if amp == torch.float16 else -6)
    for a, b in zip(grads, want_grads):
        assert (a.double() - b.double()).norm() <= bar * b.double().norm()
