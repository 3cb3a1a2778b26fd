"""The loss averaged over the tokens in the launch that forms it: statistics to the bit those of the per-token launches, the mean
against float64, the gradient to the bit the one for dloss / T in every row."""
import pytest
import torch

from tests.util import randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _peers(T, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda: torch.randn((n, T), generator=g, device=DEV)  # noqa: E731
    return [rnd() * 3, rnd().abs() + 1, rnd(), (rnd() > 0).to(torch.uint8)]


@pytest.mark.parametrize("T", [1, 63, 255, 256, 257, 8192, 32768, 32769, 70001])  # 128 blocks of 256 rows: 32768
@pytest.mark.parametrize("n_peers", [0, 1, 3])
def test_mean_of_the_per_token_losses(T, n_peers):
    from cubework_amd import ops

    V = 40
    x, t = randn((T, V), torch.bfloat16, T, std=2.0, device=DEV), torch.randint(0, 2 * V, (T,), generator=torch.Generator().manual_seed(T)).to(DEV)
    peers = _peers(T, n_peers, T + 1) if n_peers else []
    local = ops.vpce_fwd_local(x, t, V)
    rows, gmax, gsum = ops.vpce_finalize_peers(local, peers) if n_peers else ops.vpce_finalize(*(s.unsqueeze(0) for s in local))
    got = [ops.vpce_mean(x, t, V, peers) for _ in range(2)]
    assert torch.equal(got[0][0], got[1][0]) and got[0][0].dim() == 0
    assert torch.equal(got[0][1], torch.stack((gmax, gsum)))
    # sums of at most 3 rows a thread (512 at 70001), 8 levels of tree, 2 partial sums a lane, 6 levels, one division: each adds at
    # most 2^-24 of the sum of magnitudes
    bound = rows.abs().double().mean() * (-(-T // 32768) + 18) * 2.0 ** -24
    assert abs(got[0][0].double() - rows.double().mean()) <= bound
    dloss = torch.tensor(3.7, device=DEV)
    want = ops.vpce_bwd(x, t, V, gmax, gsum, (dloss.expand(T) * (1.0 / T)).contiguous())
    assert torch.equal(ops.vpce_mean_bwd(x, t, V, got[0][1], dloss), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("V", [7, 1001, 4104])
def test_mean_over_rows_of_any_type_and_pitch(V, dtype):
    from cubework_amd import ops

    T = 130
    x = randn((T, V + 3), dtype, V, std=2.0, device=DEV)[:, 1:V + 1]
    t = torch.randint(0, V, (2, T // 2), generator=torch.Generator().manual_seed(V)).to(DEV)
    a, b = x.detach().requires_grad_(True), x.detach().double().cpu().requires_grad_(True)
    loss, stats = ops.vpce_mean(a.detach(), t, 0)
    ref = torch.nn.functional.cross_entropy(b, t.reshape(-1).cpu())
    ref.backward()
    assert abs(loss.double().cpu() - ref.detach()) <= 2e-6 * ref.detach().abs()
    grad = ops.vpce_mean_bwd(x, t, 0, stats, torch.ones((), device=DEV))
    assert grad.dtype == dtype and grad.is_contiguous()
    scale = {torch.float32: 2.0 ** -20, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert (grad.double().cpu() - b.grad).abs().max() <= scale * b.grad.abs().max()


def test_no_tokens_and_wrong_targets():
    from cubework_amd.distributed import initialize
    from cubework_amd.module.loss import VocabParallelCrossEntropyLoss1D

    initialize("1d", 1)
    loss_fn = VocabParallelCrossEntropyLoss1D()
    none = loss_fn(torch.zeros((0, 8), device=DEV, requires_grad=True), torch.zeros((0,), dtype=torch.int64, device=DEV))
    assert none.dim() == 0 and torch.isnan(none)
    with pytest.raises(ValueError):
        loss_fn(torch.zeros((3, 8), device=DEV), torch.zeros((2,), dtype=torch.int64, device=DEV))


def test_a_slice_whose_peers_are_missing_is_refused():
    """Statistics staged as nothing are no statistics: not the loss of one slice alone."""
    from cubework_amd.distributed import ParallelManager as pm
    from cubework_amd.distributed import initialize
    from cubework_amd.module.loss import VocabParallelCrossEntropyLoss1D

    initialize("1d", 2, rank=1)
    x, t = torch.zeros((3, 8), device=DEV), torch.zeros((3,), dtype=torch.int64, device=DEV)
    for staged in ([], _peers(3, 1, 1)[:3]):
        pm.PARALLEL_1D.stage("vpce_stats", staged)
        with pytest.raises(ValueError):
            VocabParallelCrossEntropyLoss1D()(x, t)
    initialize("1d", 1)


def test_replays_from_a_graph():
    """The arrival count starts at zero on every replay."""
    from cubework_amd import ops

    x, t = randn((1000, 300), torch.float32, 1, device=DEV), torch.randint(0, 300, (1000,), generator=torch.Generator().manual_seed(2)).to(DEV)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        ops.vpce_mean(x, t, 0)
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        loss, stats = ops.vpce_mean(x, t, 0)
    for k in range(4):
        x.copy_(randn((1000, 300), torch.float32, 10 + k, device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        want = ops.vpce_mean(x, t, 0)
        assert torch.equal(loss, want[0]) and torch.equal(stats, want[1])
