"""What the exchanges of a larger grid deliver, added and gathered inside the kernels, against the same numbers composed with
torch (to the bit: the same fp32 additions in the same order, the same single rounding), on every kernel family and for operands
that the kernels leave to torch."""
import pytest
import torch

from tests.util import rand_uniform, randn

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _scattered(own, peers, world, rank, dtype):
    total = own
    for t in peers:
        total = total + t
    return torch.chunk(total, world, dim=-1)[rank].contiguous().to(dtype)


@pytest.mark.parametrize("shape,world", [((1, 8), 2), ((33, 520), 2), ((300, 1000), 2), ((257, 1024), 4), ((64, 2048), 8),
                                         ((9, 4096), 2), ((3, 8208), 3), ((5, 24), 3), ((7, 18), 9)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_layernorm_exchanges(shape, world, dtype):
    """world = 9 has more peers than the kernels take: torch adds and gathers them."""
    from cubework_amd import ops

    R, C = shape
    rank, H = world - 1, world * C
    x, dy = randn(shape, dtype, 1, device=DEV), randn(shape, dtype, 2, device=DEV)
    gammas = [rand_uniform((C // world,), dtype, 3 + k, 0.9, 1.1, device=DEV) for k in range(world)]
    betas = [randn((C // world,), dtype, 20 + k, 0.02, device=DEV) for k in range(world)]
    stats, gamma, beta = ops.ln_partial_stats_gather(x, gammas, betas)
    assert torch.equal(stats, ops.ln_partial_stats(x))
    assert torch.equal(gamma, torch.cat(gammas)) and torch.equal(beta, torch.cat(betas))
    others = [ops.ln_partial_stats(randn(shape, torch.float32, 40 + k, device=DEV)) for k in range(world - 1)]
    total = stats
    for t in others:
        total = total + t
    for got, want in zip(ops.ln_normalize(x, stats, H, 1e-5, gamma, beta, peers=others), ops.ln_normalize(x, total, H, 1e-5, gamma, beta)):
        assert torch.equal(got, want)
    mr = ops.ln_normalize(x, total, H, 1e-5, gamma, beta)[1]
    sums, pending = ops.ln_bwd_partials_open(dy, x, mr, gamma)
    row_peers = [randn((R, 2), torch.float32, 60 + k, device=DEV) for k in range(world - 1)]
    dgs, dbs = ([randn((C,), torch.float32, s + k, device=DEV) for k in range(world - 1)] for s in (80, 100))
    total = sums
    for t in row_peers:
        total = total + t
    dx, dg, db = ops.ln_bwd_dx_close(dy, x, mr, total, H, pending, gamma)
    for out in (dtype, torch.float32):
        got = ops.ln_bwd_dx_close(dy, x, mr, sums, H, pending, gamma, row_peers=row_peers, scatter=(dgs, dbs, world, rank, out, out))
        assert torch.equal(got[0], dx)
        assert torch.equal(got[1], _scattered(dg, dgs, world, rank, out)) and torch.equal(got[2], _scattered(db, dbs, world, rank, out))


@pytest.mark.parametrize("shape,world", [((1, 8), 2), ((300, 1000), 2), ((257, 1026), 3), ((4100, 520), 8), ((70, 18), 9)])
@pytest.mark.parametrize("activation", [None, "gelu_tanh", "relu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_bias_gradient_exchange(shape, world, activation, dtype):
    from cubework_amd import ops

    dy, pre = randn(shape, dtype, 1, device=DEV), randn(shape, dtype, 2, device=DEV)
    peers = [randn((shape[1],), torch.float32, 3 + k, device=DEV) for k in range(world - 1)]
    dpre, own = (None, ops.colsum(dy)) if activation is None else ops.act_bwd_colsum(activation, dy, pre)
    for rank in {0, world - 1}:
        got_pre, got = ops.colsum_scattered(dy, peers, world, rank, dtype, activation, pre if activation else None)
        assert torch.equal(got, _scattered(own, peers, world, rank, dtype))
        assert got_pre is None if activation is None else torch.equal(got_pre, dpre)


def test_peers_that_torch_adds():
    """Strided and 16-bit peers, a stacked tensor of them, plain numbers, a width that the ranks do not divide, no rows."""
    from cubework_amd import ops

    x = randn((40, 30), torch.bfloat16, 1, device=DEV)
    stats = ops.ln_partial_stats(x)
    odd = [torch.stack((stats, stats), 2)[..., 0], stats.bfloat16(), 3.0]
    assert not odd[0].is_contiguous()
    for peers in (odd[:1], odd[1:2], odd, torch.stack((stats, stats))):
        total = stats
        for t in peers:
            total = total + t
        assert torch.equal(ops.ln_normalize(x, stats, 90, 1e-5, peers=peers)[0], ops.ln_normalize(x, total, 90, 1e-5)[0])
    own = ops.colsum(x)
    assert torch.equal(ops.colsum_scattered(x, [own, own, own], 4, 3, torch.float16)[1], _scattered(own, [own] * 3, 4, 3, torch.float16))
    assert torch.equal(ops.colsum_scattered(x, [own], 2, 1, torch.float64)[1], _scattered(own, [own], 2, 1, torch.float64))
    dy = randn((40, 30), torch.bfloat16, 2, device=DEV)
    mr = ops.ln_normalize(x, stats, 90, 1e-5)[1]
    sums, pending = ops.ln_bwd_partials_open(dy, x, mr)
    dx, dg, db = ops.ln_bwd_dx_close(dy, x, mr, sums, 90, pending)
    for numbers in ([3.0], [own, 2], [0.25, own.bfloat16()]):
        world = len(numbers) + 1
        assert torch.equal(ops.colsum_scattered(x, numbers, world, 0, torch.bfloat16)[1], _scattered(own, numbers, world, 0, torch.bfloat16))
        got = ops.ln_bwd_dx_close(dy, x, mr, sums, 90, pending, scatter=(numbers, [own] * len(numbers), world, 0, torch.bfloat16, torch.float32))
        assert torch.equal(got[0], dx) and torch.equal(got[1], _scattered(dg, numbers, world, 0, torch.bfloat16))
        assert torch.equal(got[2], _scattered(db, [own] * len(numbers), world, 0, torch.float32))
        shifted = ops.ln_bwd_dx_close(dy, x, mr, sums, 90, pending, row_peers=[2.0])
        assert torch.equal(shifted[0], ops.ln_bwd_dx_close(dy, x, mr, sums + 2.0, 90, pending)[0])
    none = ops.colsum_scattered(x[:0], [own], 2, 0, torch.float32)[1]
    assert torch.equal(none, own[:15])
    w = [randn((15,), torch.bfloat16, 5, device=DEV), randn((15,), torch.float32, 6, device=DEV)]
    got = ops.ln_partial_stats_gather(x, w, w)
    assert torch.equal(got[1], torch.cat(w)) and torch.equal(got[0], stats)
    assert ops.ln_partial_stats_gather(x[:0], w, w)[0].shape == (0, 2)
