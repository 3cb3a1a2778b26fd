"""LayerNorm of few rows: the forward with a wavefront a chunk and the backward that finishes everything in one launch, at the edges of
their rules and of their tiles, against float64."""
import ctypes

import pytest
import torch

from tests.util import randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.bfloat16: 0, torch.float32: 1, torch.float16: 2}
# one rounding of the result, and fp32 sums of up to 4096 terms in chains of 64 and trees
REL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -18}


def _reference(x, dy, g, b, add, eps):
    x, dy, g, b, add = (t.double() for t in (x, dy, g, b, add))
    mean = x.mean(1, keepdim=True)
    rstd = (x.var(1, unbiased=False, keepdim=True) + eps).rsqrt()
    xh = (x - mean) * rstd
    gd = dy * g
    dx = (gd - gd.mean(1, keepdim=True) - xh * (gd * xh).mean(1, keepdim=True)) * rstd
    return xh * g + b, dx + add, (dy * xh).sum(0), dy.sum(0)


def _close(got, want, rel, scale=None):
    scale = want.abs() + want.abs().mean() if scale is None else scale
    assert ((got.double() - want).abs() <= rel * scale).all()


SHAPES = [(512, 768), (513, 768), (1024, 1280), (1025, 1280), (1280, 2048), (1281, 2048), (1280, 2560), (1281, 2560), (1536, 3072), (1537, 3072),
          (1792, 4096), (1793, 4096), (1, 8), (2, 520), (7, 768), (8, 1032), (9, 1536), (63, 2056), (64, 4096), (65, 1024), (257, 2048), (512, 4096), (513, 4096), (640, 768),
          (641, 768), (819, 2560), (820, 2560), (1024, 2048), (1025, 2048), (1365, 776), (1366, 776), (1536, 2048), (1537, 2048), (1792, 2560),
          (1793, 2560)]


@pytest.mark.parametrize("R,C", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("pitched", [False, True])
def test_few_rows_forward_and_backward(R, C, dtype, pitched):
    from cubework_amd import ops

    def rows(seed):
        t = randn((R, C + (64 if pitched else 0)), dtype, seed, device=DEV)
        return t[:, :C]
    x, dy, add = rows(1), rows(2), rows(3)
    g, b = (randn((C,), torch.float32, 4) * 0.2 + 1).to(dtype).to(DEV), randn((C,), dtype, 5, device=DEV)
    y, dx, dg, db = _reference(x, dy, g, b, add, 1e-5)
    got, mean_rstd = ops.ln_forward_fused(x, 1e-5, g, b)
    _close(got, y, REL[dtype])
    got_dx, got_dg, got_db = ops.ln_backward_fused(dy, x, mean_rstd, g, param_dtype=torch.float32, dx_addend=add)
    _close(got_dx, dx, REL[dtype] * 2)
    # x_hat is off by some 2^-22 of (|x - mean| + the row's largest |x|, which rounds the mean) times rstd, its sums over R rows by 2^-20 of
    # their magnitudes: 2^-19 of both
    xd = x.double()
    centred = (xd - xd.mean(1, keepdim=True)).abs() + xd.abs().amax(1, keepdim=True)
    bound = (dy.double().abs() * centred * (xd.var(1, unbiased=False, keepdim=True) + 1e-5).rsqrt()).sum(0)
    _close(got_dg, dg, 2.0 ** -19, bound)
    _close(got_db, db, 2.0 ** -20, dy.double().abs().sum(0))
    plain = ops.ln_backward_fused(dy, x, mean_rstd, g, param_dtype=dtype)
    _close(plain[0], dx - add.double(), REL[dtype] * 2)
    # without the residual gradient another kernel may take the rows: the sums' own bounds, and half a unit of their type
    unit = 0 if dtype == torch.float32 else torch.finfo(dtype).eps / 2
    assert plain[1].dtype == dtype
    _close(plain[1], dg, 1.0, 2.0 ** -19 * bound + unit * 1.001 * dg.abs())
    _close(plain[2], db, 1.0, 2.0 ** -20 * dy.double().abs().sum(0) + unit * 1.001 * db.abs())


def _backward(dy, x, mean_rstd, g, dx, ws_bytes):
    from cubework_amd import _lib
    R, C = x.shape
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    row_sums, out = torch.empty((R, 2), device=DEV), [torch.full((C,), float("nan"), device=DEV) for _ in range(2)]
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=DEV)
    rc = _lib.load().cw_ln_backward_fused(R, C, p(dy), C, p(x), C, p(mean_rstd), p(g), p(row_sums), p(dx), C, None, 0, p(out[0]), p(out[1]), 1, p(ws),
                                          ws_bytes, CODE[x.dtype], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return rc, row_sums, out


def test_in_place_and_scratch():
    """dx in the place of dY: the kernels that read every row once. Less scratch than the entry point asks for: refused as before."""
    from cubework_amd import _lib, ops
    R, C = 96, 1024
    x, dy, g = randn((R, C), torch.float32, 1, device=DEV), randn((R, C), torch.float32, 2, device=DEV), randn((C,), torch.float32, 3, device=DEV)
    _, mean_rstd = ops.ln_forward_fused(x, 1e-5, g, g)
    need = _lib.load().cw_colsum_workspace_bytes(R, C)
    dx = torch.empty_like(x)
    rc, sums, cols = _backward(dy, x, mean_rstd, g, dx, need)
    assert rc == 0
    own = dy.clone()
    rc, own_sums, own_cols = _backward(own, x, mean_rstd, g, own, need)
    assert rc == 0
    for a, b in zip([dx, sums] + cols, [own, own_sums] + own_cols):
        _close(a, b.double(), 2.0 ** -18, b.double().abs() + b.double().abs().mean())
    assert _backward(dy, x, mean_rstd, g, dx, 16)[0] == -1


@pytest.mark.parametrize("C", [512, 776, 1536, 2048, 2056, 2560, 3072, 3584, 4096])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("mode", ["one_pass", "two_pass"])
def test_a_row_has_the_same_bits_in_any_batch(C, dtype, mode):
    """On both sides of the number of rows from which a row is one wavefront's, and on the block's edges: what the ordered products
    behind the layer keep (test_forward_rows_do_not_depend_on_the_batch) begins here."""
    from cubework_amd import _lib, ops
    mode = _lib.CW_LN_ONE_PASS if mode == "one_pass" else _lib.CW_LN_TWO_PASS
    chunks = -(-C * torch.empty((), dtype=dtype).element_size() // 1024)
    edge = 4096 // chunks
    x, g, b = randn((edge + 9, C), dtype, 1, device=DEV) + 0.5, randn((C,), dtype, 2, device=DEV), randn((C,), dtype, 3, device=DEV)
    want = ops.ln_forward_fused(x, 1e-5, g, b, mode)
    for R in (1, 2, 7, 128, edge, edge + 1):
        for got, whole in zip(ops.ln_forward_fused(x[:R], 1e-5, g, b, mode), want):
            assert torch.equal(got, whole[:R])


@pytest.mark.parametrize("R,C", [(128, 1024), (700, 1024), (1536, 2048), (1537, 2048), (300, 4096)])
def test_residual_gradient_of_an_fp32_stream(R, C):
    """Added in the kernel in place of a launch behind it: the same sum but for one rounding, where the multiplication before it and the
    addition are fused (on each kernel that takes it)."""
    from cubework_amd import ops
    x, dy, add, g = (randn(s, torch.float32, k, device=DEV) for k, s in enumerate(((R, C), (R, C), (R, C), (C,))))
    _, mean_rstd = ops.ln_forward_fused(x, 1e-5, g, g)
    plain, got = (ops.ln_backward_fused(dy, x, mean_rstd, g, dx_addend=a) for a in (None, add))
    want = plain[0] + add
    assert ((got[0].double() - want.double()).abs() <= 2.0 ** -24 * (plain[0].double().abs() + 2 * want.double().abs())).all()
    assert torch.equal(got[1], plain[1]) and torch.equal(got[2], plain[2])
