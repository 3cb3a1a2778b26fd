"""Vocab-parallel cross-entropy operator: one rank's share of
_VocabParallelCrossEntropy1D/2D/3D (cubework/module/loss/loss_1d.py:11-79,
loss_2d.py:30-93, loss_3d.py:36-91).

forward: one online pass over the local logits slice gives (max, sum-exp,
target logit, mask); the MAX / SUM / SUM all-reduces of the reference
(loss_1d.py:18,44,50) become one exchange of those four per-row values, which
cw_vpce_finalize combines. backward recomputes the softmax from the saved
logits and the global (max, sum) instead of keeping a softmax-sized buffer,
and never writes into the caller's logits (the reference's 1D variant does,
loss_1d.py:20,47-48).
"""
import torch

from ... import ops
from .._amp import bwd, loss_fwd


class _VocabParallelCrossEntropy(torch.autograd.Function):

    @staticmethod
    @loss_fwd()
    def forward(ctx, logits, targets, parallel_mode):
        vocab = logits.size(-1)
        vocab_start = parallel_mode.local_rank * vocab
        logits_2d = logits.reshape(-1, vocab)
        local = ops.vpce_fwd_local(logits_2d, targets.reshape(-1), vocab_start)
        if parallel_mode.world_size == 1:
            loss, gmax, gsum = ops.vpce_finalize(*(s.unsqueeze(0) for s in local))
        else:
            # peers' (max, sumexp, pred, mask), each [world_size - 1, tokens]
            loss, gmax, gsum = ops.vpce_finalize_peers(local, parallel_mode.take("vpce_stats"))
        ctx.save_for_backward(logits_2d, targets.reshape(-1), gmax, gsum)
        ctx.meta = (vocab_start, logits.shape)
        return loss.reshape(targets.shape)

    @staticmethod
    @bwd()
    def backward(ctx, output_grad):
        logits_2d, targets, gmax, gsum = ctx.saved_tensors
        vocab_start, shape = ctx.meta
        grad = ops.vpce_bwd(logits_2d, targets, vocab_start, gmax, gsum, output_grad.reshape(-1).float(), 1.0)
        return grad.reshape(shape), None, None


class _VocabParallelCrossEntropyMean(torch.autograd.Function):
    """The loss averaged over the tokens (loss_1d.py:90-91): the launch that forms the losses finishes their mean, and the gradient
    kernel reads the mean's gradient."""

    @staticmethod
    @loss_fwd()
    def forward(ctx, logits, targets, vocab_start, peers):
        logits_2d, targets = logits.reshape(-1, logits.size(-1)), targets.reshape(-1)
        loss, stats = ops.vpce_mean(logits_2d, targets, vocab_start, peers)
        ctx.save_for_backward(logits_2d, targets, stats)
        ctx.meta = (vocab_start, logits.shape)
        return loss

    @staticmethod
    @bwd()
    def backward(ctx, output_grad):
        logits_2d, targets, stats = ctx.saved_tensors
        vocab_start, shape = ctx.meta
        return ops.vpce_mean_bwd(logits_2d, targets, vocab_start, stats, output_grad).reshape(shape), None, None, None


def vocab_parallel_cross_entropy(logits, targets, parallel_mode):
    """Per-token loss [targets.shape] for this rank's vocabulary slice."""
    return _VocabParallelCrossEntropy.apply(logits, targets, parallel_mode)


def vocab_parallel_cross_entropy_mean(logits, targets, parallel_mode):
    """Mean loss over the tokens for this rank's vocabulary slice."""
    if targets.numel() == 0:  # a mean of nothing: NaN, as torch gives it
        return _VocabParallelCrossEntropy.apply(logits, targets, parallel_mode).mean()
    vocab_start = parallel_mode.local_rank * logits.size(-1)
    peers = ()
    if parallel_mode.world_size > 1:
        peers = parallel_mode.take("vpce_stats")
        if len(peers) != 4:  # none at all would be a slice without peers to the operator
            raise ValueError("the peers' max, sumexp, pred and mask are needed")
    loss = ops.mean_loss(logits, targets, vocab_start, peers)
    return _VocabParallelCrossEntropyMean.apply(logits, targets, vocab_start, peers) if loss is None else loss
