"""Vocab-parallel cross-entropy over rows of any alignment: row lengths around the vector and batch sizes, pitches and
start addresses that put every row at another offset, gradients with padded rows; against the oracle in float64."""
import pytest
import torch

from tests.util import assert_parity, randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _place(t, pitch, start):
    """t [T, V] on the device with the given row pitch, `start` elements into its buffer, NaN around it."""
    T, V = t.shape
    buf = torch.full((start + T * pitch,), float("nan"), dtype=t.dtype, device=DEV)
    view = buf[start:].view(T, pitch)[:, :V]
    view.copy_(t)
    return view


@pytest.mark.parametrize("V", [1, 3, 7, 8, 9, 250, 2047, 6145, 8195, 12571])
@pytest.mark.parametrize("dtype,grad_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                              (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("extra,start", [(0, 0), (1, 0), (0, 1), (2, 3)])
def test_rows_of_any_alignment(V, dtype, grad_dtype, extra, start):
    import oracle
    from cubework_amd import ops

    T = 5
    x = randn((T, V), dtype, seed=V, std=2.0)
    t = torch.tensor([V, V + V - 1, 0, V + V // 2, 2 * V])  # first, last, before, inside, past the slice
    dl = torch.linspace(0.5, 1.5, T)
    view = _place(x, V + extra, start)
    got = ops.vpce_fwd_local(view, t.to(DEV), V)
    loss, gmax, gsum = ops.vpce_finalize(*(g.unsqueeze(0) for g in got))
    grads = [ops.vpce_bwd(view, t.to(DEV), V, gmax, gsum, dl.to(DEV), 1.0, grad_dtype=grad_dtype, aligned_rows=a) for a in (False, True)]
    with oracle.precision(torch.float64):
        want = oracle.vpce_fwd_local(x, t, V)
        want_grad = oracle.vpce_bwd(x, t, V, gmax.cpu(), gsum.cpu(), dl)
    what = "V=%d %s extra=%d start=%d" % (V, dtype, extra, start)
    assert torch.equal(got[0].cpu(), want[0].float()) and torch.equal(got[2].cpu(), want[2].float())
    assert torch.equal(got[3].cpu(), want[3])
    assert_parity(got[1], want[1], torch.float32, "sum exp " + what)
    assert grads[0].is_contiguous() and torch.equal(grads[0], grads[1])
    assert T == 1 or grads[1].stride(0) * grads[1].element_size() % 16 == 0
    assert_parity(grads[0], want_grad, grad_dtype, "gradient " + what)


@pytest.mark.parametrize("V", [1001, 1000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_head_gradients_with_padded_rows(V, dtype):
    """The classifier's two gradient products from the loss's contiguous gradient and from one that a hook returns with padded rows."""
    from cubework_amd.distributed import initialize
    from cubework_amd.module.loss import VocabParallelCrossEntropyLoss1D
    from cubework_amd.module.parallel_1d import VocabParallelClassifier1D

    initialize("1d", 1)
    with torch.device(DEV):
        layer = VocabParallelClassifier1D(96, V, bias=True).to(dtype)
    loss_fn = VocabParallelCrossEntropyLoss1D()
    targets = torch.randint(0, V, (2, 61), generator=torch.Generator().manual_seed(1)).to(DEV)
    results = []

    def padded(g):
        out = torch.full(g.shape[:-1] + (V + 15,), float("nan"), dtype=dtype, device=DEV)[..., :V]
        return out.copy_(g)

    for contiguous in (False, True):
        x = randn((2, 61, 96), dtype, seed=2).to(DEV).requires_grad_(True)
        layer.zero_grad()
        logits = layer(x)
        if not contiguous:
            logits.register_hook(padded)
        loss_fn(logits, targets).backward()
        results.append([x.grad] + [p.grad.clone() for p in layer.parameters()])
    for got, want in zip(*results):
        # the same products from other addresses: the 16-bit kernel copies unaligned rows and multiplies the same values,
        # the fp32 one may take another kernel and so another order of its sums
        assert_parity(got, want.cpu(), dtype, "head gradient V=%d" % V)


@pytest.mark.parametrize("T", [1, 255, 257, 8192])
@pytest.mark.parametrize("n_peers", [0, 1, 3])
def test_finalize_from_the_peers_as_they_arrived(T, n_peers):
    """The same combination as of the stacked statistics, in the same order: the same bits. A rank without a finite logit
    and peers of another type are among them."""
    from cubework_amd import ops

    g = torch.Generator(device=DEV).manual_seed(T + n_peers)
    rnd = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    stats = [rnd(n_peers + 1, T) * 3, rnd(n_peers + 1, T).abs() + 1, rnd(n_peers + 1, T), torch.ones(n_peers + 1, T, dtype=torch.uint8, device=DEV)]
    stats[0][-1, 0], stats[1][-1, 0] = float("-inf"), 0.0
    stats[3][torch.arange(T, device=DEV) % (n_peers + 1), torch.arange(T, device=DEV)] = 0
    want = ops.vpce_finalize(*stats)
    peers = [s[1:].double() if k < 3 else s[1:].bool() for k, s in enumerate(stats)]
    got = ops.vpce_finalize_peers([s[0].contiguous() for s in stats], peers)
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("V", [1001, 1000])
def test_logits_gradient_is_contiguous(V):
    """Hooks on the logits and retain_grad see a dense gradient for every vocabulary, as any operator's."""
    from cubework_amd.distributed import initialize
    from cubework_amd.module.loss import VocabParallelCrossEntropyLoss1D
    from cubework_amd.module.parallel_1d import VocabParallelClassifier1D

    initialize("1d", 1)
    with torch.device(DEV):
        layer = VocabParallelClassifier1D(96, V, bias=False).to(torch.bfloat16)
    x = randn((2, 61, 96), torch.bfloat16, seed=2).to(DEV).requires_grad_(True)
    logits = layer(x)
    seen = []
    logits.register_hook(lambda g: seen.append(g.view(-1).numel()))
    logits.retain_grad()
    VocabParallelCrossEntropyLoss1D()(logits, torch.zeros((2, 61), dtype=torch.int64, device=DEV)).backward()
    assert seen == [2 * 61 * V] and logits.grad.is_contiguous() and logits.grad.untyped_storage().nbytes() == 2 * 61 * V * 2


@pytest.mark.parametrize("V", [1, 2, 7, 9, 767, 769, 4095, 4097, 6143, 6145, 8191, 8193, 16384])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_cross_entropy_of_odd_rows(V, dtype):
    """Rows at every alignment of their elements, in both kernels: vectors from the first or the second element on."""
    from cubework_amd import ops

    T = 5
    for first in (0, 1):
        buf = randn((T * V + 1,), dtype, V, std=3.0, device=DEV)
        x = buf[first:first + T * V].view(T, V)
        t = torch.tensor([0, V - 1, min(1, V - 1), V // 2, V + 3], device=DEV)  # the last one: another slice's
        m, s, p, k = ops.vpce_fwd_local(x, t, 0)
        ref = x.double()
        top = ref.max(1).values
        assert torch.equal(m.double(), top) and k.tolist() == [0, 0, 0, 0, 1]
        # exponentials to 2^-22 or so, V terms at most 2^-24 each in chains of V / 2048 + 32
        want = (ref - top[:, None]).exp().sum(1)
        assert ((s.double() - want).abs() <= (V / 2048 + 40) * 2.0 ** -23 * want).all()
        assert torch.equal(p[:4], x[torch.arange(4), t[:4]].float()) and p[4] == 0
        soft = (ref - top[:, None]).exp() / want[:, None]
        soft[torch.arange(4), t[:4]] -= 1.0
        for aligned in (False, True):
            g = ops.vpce_bwd(x, t, 0, m, s, aligned_rows=aligned)
            rel = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
            assert ((g.double() - soft).abs() <= rel * soft.abs() + 2.0 ** -20 * (1 if dtype == torch.bfloat16 else 2.0 ** -4)).all()
