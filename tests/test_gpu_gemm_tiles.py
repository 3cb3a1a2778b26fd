"""GPU parity of the tile kernels of the 16-bit block GEMM against the CPU oracle where they can go wrong: edges and
remainders of every tile size, reduction lengths that end inside a 16-byte chunk, sliced reductions, operands and addends
with unaligned rows (copied), unaligned output rows, more k-steps than one trip holds."""
import pytest
import torch

from tests.util import assert_parity, randn

pytestmark = pytest.mark.gpu

# (M, N, K, steps): below one tile, one element past a tile, K inside a chunk / a k block, many tiles of each size
SHAPES = [(1, 1, 1, 1), (3, 5, 7, 1), (64, 64, 32, 1), (65, 63, 33, 2), (128, 129, 31, 1), (127, 256, 72, 3), (257, 255, 64, 1),
          (77, 1001, 1003, 1), (300, 4096, 136, 1), (64, 768, 3072, 1), (130, 520, 4100, 2), (1554, 776, 72, 1), (4352, 4104, 40, 1)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("layout", ["NN", "NT", "TN"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_edges_of_every_tile(layout, shape, dtype):
    import oracle
    from cubework_amd import ops

    M, N, K, steps = shape
    a_shape, b_shape = ((K, M) if layout == "TN" else (M, K)), ((N, K) if layout == "NT" else (K, N))
    A = [randn(a_shape, dtype, 3 * i) for i in range(steps)]
    B = [randn(b_shape, dtype, 3 * i + 1, std=0.05) for i in range(steps)]
    bias, add = randn((N,), dtype, 90), [randn((M, N), dtype, 91), randn((M, N), dtype, 92)]
    act = None if layout == "TN" else "gelu_erf"
    # fp32 sums of up to 2 x 4100 products rounded once: the storage type's bar
    want = oracle.gemm_ksteps(layout, A, B, bias, act, add)
    got = ops.gemm_ksteps(layout, [a.cuda() for a in A], [b.cuda() for b in B], bias.cuda(), act, [t.cuda() for t in add])
    assert_parity(got, want, dtype, "%s %s %s" % (layout, shape, dtype))


@pytest.mark.parametrize("layout", ["NN", "NT", "TN"])
def test_unaligned_views_and_many_steps(layout):
    """Every operand a view with an odd row pitch and base, six k-steps, a padded output."""
    import oracle
    from cubework_amd import ops

    M, N, K, steps = 133, 267, 70, 6
    a_shape, b_shape = ((K, M) if layout == "TN" else (M, K)), ((N, K) if layout == "NT" else (K, N))

    def view(shape, seed, std=1.0):
        return randn((shape[0], shape[1] + 5), torch.bfloat16, seed, std).cuda()[:, 3:3 + shape[1]]
    A, B = [view(a_shape, 2 * i) for i in range(steps)], [view(b_shape, 2 * i + 1, 0.05) for i in range(steps)]
    add = [view((M, N), 50)]
    out = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device="cuda")
    got = ops.gemm_ksteps(layout, A, B, None, None, add, out=out[:, :N])
    want = oracle.gemm_ksteps(layout, [a.cpu() for a in A], [b.cpu() for b in B], None, None, [t.cpu() for t in add])
    assert_parity(got, want, torch.bfloat16, "unaligned %s" % layout)
    assert (out[:, N:] == 7.0).all()


def test_rows_beside_a_nan_stay_finite():
    """A NaN behind the last column of a reduction that ends inside a chunk must not reach the result."""
    import oracle
    from cubework_amd import ops

    M, N, K = 200, 136, 77
    parent = randn((M, 80), torch.bfloat16, 1)
    parent[:, K:] = float("nan")
    a, b = parent[:, :K], randn((K, N), torch.bfloat16, 2, 0.05)
    assert_parity(ops.gemm_ksteps("NN", [parent.cuda()[:, :K]], [b.cuda()]), oracle.gemm_ksteps("NN", [a], [b]), torch.bfloat16, "nan beside K")


def test_forward_rows_do_not_depend_on_the_batch():
    """A projection's row has the same bits whatever rows stand beside it (k is summed in one order)."""
    from cubework_amd import ops

    a, b = randn((900, 1024), torch.float16, 1).cuda(), randn((1024, 1024), torch.float16, 2, 0.02).cuda()
    whole = ops.gemm_ksteps("NN", [a], [b])
    for rows in (1, 65, 300):
        assert torch.equal(ops.gemm_ksteps("NN", [a[:rows]], [b]), whole[:rows])
