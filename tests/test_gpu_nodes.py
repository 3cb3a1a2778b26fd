"""The native autograd nodes against the Python ones: the same launches, so the same bits, forward and backward, over the forms of
operands that both take; and the calls that stay with the Python nodes."""
import contextlib

import pytest
import torch

from tests.util import randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _modes():
    from cubework_amd.distributed import initialize, pm
    initialize("2d", 1)
    return pm.PARALLEL_2D_ROW, pm.PARALLEL_2D_COL


def _x(shape, dtype, seed, form):
    if form == "strided":
        return randn(shape[:-1] + (2 * shape[-1],), dtype, seed, device=DEV)[..., ::2]
    if form == "offset":
        return randn((shape[0] + 1,) + shape[1:], dtype, seed, device=DEV)[1:]
    return randn(shape, dtype, seed, device=DEV)


def _compare(native, python, leaves, dy):
    """Outputs and gradients of two ways to run the same operator on clones of the same leaves."""
    results = []
    for fn in (native, python):
        own = [None if t is None else t.detach().clone(memory_format=torch.preserve_format).requires_grad_(t.requires_grad) for t in leaves]
        out = fn(*own)
        out = out if isinstance(out, tuple) else (out,)
        torch.autograd.backward(out, [dy(o, k) for k, o in enumerate(out)])
        results.append([o.detach() for o in out] + [None if t is None else t.grad for t in own])
    for a, b in zip(*results):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
    return results[0]


def _dy(o, k):
    return randn(tuple(o.shape), o.dtype, 90 + k, device=DEV) if k == 0 else torch.ones_like(o)


AMP = {None: contextlib.nullcontext, "fp16": lambda: torch.autocast("cuda"), "bf16": lambda: torch.autocast("cuda", dtype=torch.bfloat16)}


@pytest.mark.parametrize("amp", [None, "fp16", "bf16"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape,form", [((5, 24), "plain"), ((3, 7, 40), "plain"), ((40,), "plain"), ((6, 40), "strided"), ((2, 5, 44), "offset")])
@pytest.mark.parametrize("activation,bias,residual", [(None, True, True), (None, False, False), ("relu", True, False), ("gelu_tanh", True, False),
                                                      ("gelu", False, False)])
def test_linear(shape, form, dtype, amp, activation, bias, residual):
    from cubework_amd import ops
    from cubework_amd.module.parallel_1d._operation import _LinearNT
    from cubework_amd.module.parallel_2d._operation import _SUMMA_AB

    row, col = _modes()
    K, N = shape[-1], 56
    x = _x(shape, dtype, 1, form).requires_grad_(True)
    b = randn((N,), dtype, 3, device=DEV).requires_grad_(True) if bias else None
    r = randn(shape[:-1] + (N,), dtype, 4, device=DEV).requires_grad_(True) if residual else None

    def run(fn):
        def body(*leaves):
            with AMP[amp]():
                return fn(*leaves)
        return body

    w = randn((K, N), dtype, 2, 0.1, device=DEV).requires_grad_(True)
    if len(shape) == 1:
        assert ops.linear("NN", x, w) is None  # the 2D node has no backward for a vector
    else:
        _compare(run(lambda x, w, b, r: ops.linear("NN", x, w, b, activation, r)),
                 run(lambda x, w, b, r: _SUMMA_AB.apply(x, w, b, 1, shape[:-1] + (N,), row, col, activation, r)), (x, w, b, r), _dy)
    if not residual:
        w = randn((N, K), dtype, 2, 0.1, device=DEV).requires_grad_(True)
        _compare(run(lambda x, w, b: ops.linear("NT", x, w, b, activation)), run(lambda x, w, b: _LinearNT.apply(x, w, b, activation)),
                 (x, w, b), _dy)
        w.requires_grad_(False)  # a frozen weight, an expanded gradient
        got = _compare(run(lambda x, w, b: ops.linear("NT", x, w, b, activation)), run(lambda x, w, b: _LinearNT.apply(x, w, b, activation)),
                       (x, w, b), lambda o, k: torch.ones((), dtype=o.dtype, device=DEV).expand_as(o))
        assert got[2] is None


@pytest.mark.parametrize("amp", [None, "fp16"])
@pytest.mark.parametrize("dtype,pdtype", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32), (torch.float16, torch.float32)])
@pytest.mark.parametrize("shape,form", [((5, 24), "plain"), ((3, 7, 1024), "plain"), ((40,), "plain"), ((6, 44), "strided"), ((9, 12288), "offset")])
@pytest.mark.parametrize("fork", [False, True])
def test_layernorm(shape, form, dtype, pdtype, amp, fork):
    from cubework_amd import ops
    from cubework_amd.module.parallel_2d._operation import _Layernorm2D

    row, col = _modes()
    C = shape[-1]
    leaves = [_x(shape, dtype, 1, form), randn((C,), pdtype, 2, device=DEV), randn((C,), pdtype, 3, device=DEV)]
    for t in leaves:
        t.requires_grad_(True)

    def native(x, w, b):
        with AMP[amp]():
            return ops.layernorm(x, w, b, 1e-5, fork)

    def python(x, w, b):
        with AMP[amp]():
            return _Layernorm2D.apply(x, w, b, C, 1e-5, row, col, fork)

    _compare(native, python, leaves, _dy)


@pytest.mark.parametrize("d", [64, 128, 48, 80])
@pytest.mark.parametrize("scale,causal", [(None, True), (0.3, False)])
def test_attention(d, scale, causal):
    from cubework_amd import _lib, ops

    qkv = randn((2, 77, 3 * 3 * d), torch.bfloat16, 1, device=DEV).requires_grad_(True)
    _compare(lambda t: _lib.host().attention(t, 3, scale, causal), lambda t: ops._AttentionCore.apply(t, 3, scale, causal), [qkv], _dy)


@pytest.mark.parametrize("tokens,width", [((3, 50), 64), ((7,), 33), ((20000,), 8)])  # 20000: through the token order
@pytest.mark.parametrize("id_type", [torch.int64, torch.int32])
def test_embedding(tokens, width, id_type):
    from cubework_amd import _lib, ops

    ids = torch.randint(0, 120, tokens, generator=torch.Generator().manual_seed(1)).to(DEV, id_type)
    w = randn((50, width), torch.bfloat16, 2, device=DEV).requires_grad_(True)
    _compare(lambda w: _lib.host().embedding(ids, w, 30, 4), lambda w: ops._VocabEmbedding.apply(ids, w, 30, 4), [w], _dy)


@pytest.mark.parametrize("amp", [None, "fp16"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_mean_loss(dtype, amp):
    from cubework_amd import ops
    from cubework_amd.module.loss._operation import _VocabParallelCrossEntropyMean

    x = randn((2, 33, 101), dtype, 1, 2.0, device=DEV).requires_grad_(True)
    t = torch.randint(0, 202, (2, 33), generator=torch.Generator().manual_seed(2)).to(DEV)
    peers = [randn((1, 66), torch.float32, 3, device=DEV) for _ in range(3)] + [torch.zeros((1, 66), dtype=torch.uint8, device=DEV)]

    def run(fn):
        def body(x):
            with AMP[amp]():
                return fn(x)
        return body
    _compare(run(lambda x: ops.mean_loss(x, t, 101, peers)), run(lambda x: _VocabParallelCrossEntropyMean.apply(x, t, 101, peers)), [x],
             lambda o, k: torch.full_like(o, 2.5))


class _Sub(torch.Tensor):
    pass


def test_calls_that_stay_with_the_python_nodes():
    from torch.utils._python_dispatch import TorchDispatchMode

    from cubework_amd import _lib, ops
    from cubework_amd.module.parallel_1d._operation import linear_nt

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, w = randn((4, 8), torch.float32, 1, device=DEV), randn((8, 8), torch.float32, 2, device=DEV)
    assert ops.linear("NN", x, w) is not None and ops.layernorm(x, w[0], w[1], 1e-5) is not None
    refused = [lambda: ops.linear("NN", x.as_subclass(_Sub), w), lambda: ops.linear("NN", x.cpu(), w), lambda: ops.linear("NN", x, w[:4]),
               lambda: ops.linear("NN", x[:, :0], w[:0]), lambda: ops.linear("NN", x, w, None, "relu", x), lambda: ops.linear("NN", 3, w),
               lambda: ops.layernorm(x, w[0, :4], w[0], 1e-5), lambda: ops.layernorm(x.double(), w[0], w[1], 1e-5),
               lambda: ops.mean_loss(x[:0], torch.zeros(0, dtype=torch.int64, device=DEV), 0),
               lambda: _lib.host().attention(x, 1, None, True), lambda: _lib.host().embedding(x, w, 0, -1)]
    for call in refused:
        assert call() is None
    with Watch():
        assert ops.linear("NN", x, w) is None and ops.layernorm(x, w[0], w[1], 1e-5) is None
    seen = []
    torch.func.vmap(lambda t: seen.append(ops.linear("NN", t, w)) or t)(x[None])
    torch.jit.trace(lambda t: (seen.append(ops.linear("NN", t, w)), t * 2)[1], (x,), check_trace=False)
    assert seen == [None, None]
    with pytest.raises(KeyError):
        ops.linear("NN", x, w, None, "swish")
    with torch.autograd.forward_ad.dual_level():
        assert ops.linear("NN", x, w) is None
        dual = torch.autograd.forward_ad.make_dual(x, x)
        with pytest.raises(NotImplementedError):
            linear_nt(dual, w)


def test_saved_tensor_hooks_and_checkpoint():
    from torch.utils.checkpoint import checkpoint

    from cubework_amd.opt_block import OPTBlock

    _modes()
    with torch.device(DEV):
        blk = OPTBlock(hidden=128, heads=2, ffn=256, dtype=torch.bfloat16)
    x, dy = (randn((2, 40, 128), torch.bfloat16, k, device=DEV) for k in (1, 2))

    def grads(forward):
        blk.zero_grad(set_to_none=True)
        a = x.detach().clone().requires_grad_(True)
        forward(a).backward(dy)
        return [a.grad] + [p.grad for p in blk.parameters()]

    want, packed = grads(blk), []

    def hooked(a):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.to(DEV)):
            return blk(a)

    for forward in (hooked, lambda a: checkpoint(blk, a, use_reentrant=False), lambda a: checkpoint(blk, a, use_reentrant=True)):
        for got, ref in zip(grads(forward), want):
            assert torch.equal(got, ref)
    assert len(packed) >= 4 * 2 + 2 * 3 + 3


def test_modified_inputs_and_second_derivatives_are_refused():
    from cubework_amd import ops

    x, w = (randn((8, 8), torch.float32, k, device=DEV).requires_grad_(True) for k in (1, 2))
    y = ops.linear("NN", x, w)
    with torch.no_grad():
        w.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        y.sum().backward()
    (g,) = torch.autograd.grad(ops.linear("NN", x, w).sum(), x, create_graph=True)
    assert not g.requires_grad


def test_errors_of_the_library_reach_the_caller_from_the_backward_thread():
    import ctypes

    from cubework_amd import _lib, ops

    host, lib = _lib.host(), _lib.load()
    real = {n: getattr(lib, n) for n in _lib.HOST_ENTRIES}
    restype, argtypes = _lib.SIGNATURES["cw_colsum"]
    refuse = ctypes.CFUNCTYPE(restype, *argtypes)(lambda *a: _lib.CW_ERR_UNSUPPORTED)
    x, w, b = (randn(s, torch.float32, 1, device=DEV).requires_grad_(True) for s in ((8, 8), (8, 8), (8,)))
    y = ops.linear("NN", x, w, b)
    try:
        _lib.bind_host(host, {**real, "cw_colsum": refuse})
        with pytest.raises(_lib.CubeworkHipError):
            y.sum().backward()
    finally:
        _lib.bind_host(host, real)
    ops.linear("NN", x, w, b).sum().backward()
    assert b.grad is not None


def test_threads_and_streams():
    """Steps on four threads, each on a stream of its own, give what one thread gives."""
    import threading

    from cubework_amd.opt_block import OPTBlock

    _modes()
    with torch.device(DEV):
        blocks = [OPTBlock(hidden=128, heads=2, ffn=256, dtype=torch.bfloat16) for _ in range(4)]
    x, dy = (randn((1, 64, 128), torch.bfloat16, k, device=DEV) for k in (1, 2))
    torch.cuda.synchronize()

    def step(blk, out):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(5):
                blk.zero_grad(set_to_none=True)
                a = x.detach().clone().requires_grad_(True)
                y = blk(a)
                y.backward(dy)
        stream.synchronize()
        out[:] = [y.detach(), a.grad] + [p.grad for p in blk.parameters()]

    alone, together = [[] for _ in blocks], [[] for _ in blocks]
    for blk, out in zip(blocks, alone):
        step(blk, out)
    threads = [threading.Thread(target=step, args=a) for a in zip(blocks, together)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, together):
        assert len(a) == len(b) > 0 and all(torch.equal(p, q) for p, q in zip(a, b))


@pytest.mark.parametrize("rows,vocab,bias", [(33, 1001, False), (257, 516, True), (64, 1000, False), (1, 7, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_head_and_loss_of_any_vocabulary(rows, vocab, bias, dtype):
    """The head's gradients are the ones of a dense gradient of the logits, and whoever sees that gradient sees a dense one."""
    from cubework_amd import ops
    from cubework_amd.module.loss._operation import _VocabParallelCrossEntropyMean
    from cubework_amd.module.parallel_1d._operation import _LinearNT

    leaves = [randn((rows, 64), dtype, 1, device=DEV).requires_grad_(True), randn((vocab, 64), dtype, 2, std=0.1, device=DEV).requires_grad_(True),
              randn((vocab,), dtype, 3, device=DEV).requires_grad_(True) if bias else None]
    t = torch.randint(0, vocab, (rows,), generator=torch.Generator().manual_seed(4)).to(DEV)
    scale = lambda o, k: torch.full_like(o, 64.0)  # noqa: E731
    want = _compare(lambda x, w, b: ops.mean_loss(ops.linear("NT", x, w, b), t, 0),
                    lambda x, w, b: _VocabParallelCrossEntropyMean.apply(_LinearNT.apply(x, w, b, None), t, 0, ()), leaves, scale)
    x, w, b = leaves
    seen = []
    forward = lambda: ops.linear("NT", x, w, b)  # noqa: E731
    for watch in ("hook", "retain", "post", "behind", "asked", "inputs", "view"):
        for leaf in leaves:
            if leaf is not None:
                leaf.grad = None
        logits = forward()
        loss = ops.mean_loss(logits.view(rows, 1, vocab) if watch == "view" else logits, t, 0)
        dy = torch.full_like(loss, 64.0)
        if watch == "hook":
            logits.register_hook(seen.append)
        elif watch == "retain":
            logits.retain_grad()
        elif watch == "post":
            loss.grad_fn.register_hook(lambda outputs, _: seen.append(outputs[0]))
        elif watch == "behind":  # the layer's own node: its hooks are handed what it was given
            logits.grad_fn.register_hook(lambda _, given: seen.append(given[0]))
        if watch == "asked":
            seen.append(torch.autograd.grad(loss, logits, dy)[0])
            continue
        loss.backward(dy, inputs=[logits, x] if watch == "inputs" else None)
        if watch in ("retain", "inputs"):
            seen.append(logits.grad)
        assert torch.equal(x.grad, want[1])
        if watch != "inputs":
            assert torch.equal(w.grad, want[2])
    assert len(seen) == 6
    assert all(g.shape == (rows, vocab) and g.is_contiguous() and torch.equal(g, seen[0]) for g in seen)
    # the logits read a second time: their gradients are added before the product sees them
    logits = forward()
    (twice,) = torch.autograd.grad(ops.mean_loss(logits, t, 0) + logits.float().sum() / 16, x)
    ref = torch.autograd.grad(ops.mean_loss(forward(), t, 0), x)[0].double() + (w.double().sum(0) / 16)
    # 16-bit rounding of the added gradient and of the results
    assert (twice.double() - ref).abs().max() <= 2.0 ** (-7 if dtype == torch.bfloat16 else -10) * ref.abs().max()


@pytest.mark.parametrize("watch", ["hook", "retain", "asked"])
def test_residual_of_a_head_of_an_odd_vocabulary(watch):
    """A layer hands its residual the gradient it was given: a dense one, which a hook may view as it likes."""
    from cubework_amd import ops

    x, w = randn((33, 64), torch.bfloat16, 1, device=DEV).requires_grad_(True), randn((64, 1001), torch.bfloat16, 2, std=0.1, device=DEV).requires_grad_(True)
    leaf = randn((33, 1001), torch.bfloat16, 3, device=DEV).requires_grad_(True)
    t = torch.randint(0, 1001, (33,), generator=torch.Generator().manual_seed(4)).to(DEV)
    residual = leaf * 1.0
    loss = ops.mean_loss(ops.linear("NN", x, w, residual=residual), t, 0)
    seen = []
    if watch == "hook":
        residual.register_hook(lambda g: seen.append(g.view(-1)))
    elif watch == "retain":
        residual.retain_grad()
    if watch == "asked":
        seen.append(torch.autograd.grad(loss, residual)[0])
    else:
        loss.backward()
        seen.append(leaf.grad if watch == "hook" else residual.grad)
    assert len(seen) == (2 if watch == "hook" else 1) and all(g.is_contiguous() and g.numel() == 33 * 1001 for g in seen)
