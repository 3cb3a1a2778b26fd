"""Attention at head sizes that are multiples of 8 and neither 64 nor 128, which the kernels read at their own width:
every shape of the head dispatch at its smallest and largest size, at token counts around the tile edges, against the
oracle, and rows that are not 16-byte aligned, which go through the zero-padded copy."""
import pytest
import torch

from tests.util import assert_parity, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(x, heads, d_out, causal):
    from cubework_amd import ops

    x = x.detach().requires_grad_(True)
    y = ops.attention_core(x, heads, None, causal)
    y.backward(d_out)
    return y.detach(), x.grad


@pytest.mark.parametrize("d", [8, 40, 48, 56, 72, 80, 88, 120])
@pytest.mark.parametrize("shape,causal", [((2, 1, 3), True), ((1, 65, 2), True), ((2, 300, 3), True), ((1, 257, 2), False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_native_head_sizes(d, shape, causal, dtype):
    import oracle

    b, s, h = shape
    qkv = randn((b, s, h * 3 * d), dtype, seed=d + s)
    d_out = randn((b, s, h * d), dtype, seed=d + s + 1)
    y, g = _run(qkv.to(DEV), h, d_out.to(DEV), causal)
    with oracle.precision(torch.float64):
        qc, kc, vc = oracle.split_qkv(qkv, h)
        want = oracle.attention_core(qc, kc, vc, causal=causal)
        grads = oracle.attention_core_backward(qc, kc, vc, d_out, causal=causal)
    what = "%s head size %d %s causal=%s" % (dtype, d, shape, causal)
    assert_parity(y, want, dtype, "attention " + what)
    # dq and dk vanish for a single token: compared with the rest of the tensor
    assert_parity(g, torch.cat(grads, dim=-1).permute(0, 2, 1, 3).reshape(b, s, h * 3 * d), dtype, "attention dqkv " + what)


@pytest.mark.parametrize("d", [48, 80])
@pytest.mark.parametrize("form", ["rows", "pointer", "gradient"])
def test_unaligned_rows(d, form):
    b, s, h = 2, 100, 3
    w = h * 3 * d
    qkv = randn((b, s, w), torch.bfloat16, seed=d).to(DEV)
    d_out = randn((b, s, h * d), torch.bfloat16, seed=d + 1).to(DEV)
    want = _run(qkv, h, d_out, True)
    if form == "rows":
        wide = torch.full((b, s, w + 1), float("nan"), dtype=qkv.dtype, device=DEV)
        wide[..., :w] = qkv
        x = wide[..., :w]
    elif form == "pointer":
        x = torch.empty(qkv.numel() + 1, dtype=qkv.dtype, device=DEV)[1:].view(b, s, w).copy_(qkv)
    else:
        x = qkv
        d_out = torch.empty(d_out.numel() + 1, dtype=qkv.dtype, device=DEV)[1:].view(b, s, h * d).copy_(d_out)
    got = _run(x, h, d_out, True)
    for a, e in zip(got, want):
        # the padded copy adds products with zeros only; its 64 or 128 columns are the same sums
        assert_parity(a, e.float(), torch.bfloat16, "unaligned %s, head size %d" % (form, d))


@pytest.mark.parametrize("D", [48, 56, 64, 80, 96, 128])
@pytest.mark.parametrize("B,H,S,causal", [(9, 16, 130, True), (5, 16, 257, True), (5, 32, 300, False), (18, 16, 130, True), (17, 16, 260, True),
                                           (5, 32, 500, False), (16, 16, 1024, False), (16, 16, 1400, True)])
def test_blocks_of_any_number_of_wavefronts_give_the_same_bits(B, H, S, D, causal):
    """A batch on each side of the rules that choose a block's wavefronts, against its sequences one by one: whole batches run on blocks of 4
    or 8, single sequences on blocks of 2 or 4."""
    qkv, d_out = randn((B, S, H * 3 * D), torch.bfloat16, D + S, device=DEV), randn((B, S, H * D), torch.bfloat16, D, device=DEV)
    whole = _run(qkv, H, d_out, causal)
    for b in (0, B - 1):
        for one, all_of in zip(_run(qkv[b:b + 1].contiguous(), H, d_out[b:b + 1].contiguous(), causal), whole):
            assert torch.equal(one, all_of[b:b + 1])
