"""GPU parity of the block GEMM's kernels of 8 wavefronts (256-column tiles, 128 x 128 tiles with two groups of wavefronts
along k, 128-column tiles of up to 192 rows: configurations 0 and 5 to 7 of the planner) against float64 where they can go wrong:
every tile height, edges of M and N, steps whose K ends inside a stage, units of no more stages than the kernel takes, seams of steps
and of tiles, sliced tiles, unaligned output rows, every operand of the epilogue. Which configuration the planner gives a shape in
which orientation is held by tests/test_gemm_plans.py."""
import pytest
import torch

from tests.util import assert_parity, randn

pytestmark = pytest.mark.gpu

# (M, N, K, steps), which the planner gives to 256-column tiles in NN and NT and, mostly, in TN: heights 160, 192, 224 and 256 with
# ragged edges, K of a part of a stage behind whole ones, three steps (rotated starts in NT), three tiles a block, a last row and column
# of tiles with few elements, an odd last column; three stages to a tile, each of them a part of one (as short as the kernel
# takes: every stage is the last of its step, every third of its tile); slices of three and four stages (NT and TN)
SHAPES = [(300, 50257, 40, 3), (4100, 4090, 392, 1), (300, 32768, 1016, 1), (376, 32760, 1000, 1), (1552, 7672, 1352, 1), (8184, 2040, 328, 3), (8184, 6136, 520, 1),
          (7000, 4600, 1000, 1), (1024, 25003, 768, 1), (8192, 2048, 512, 2)]

# shapes that the planner gives to 128 x 128 tiles of two groups, in one orientation at least: ragged last tiles of either direction, K
# that ends in the first and in the second half of a stage, several steps, a short reduction, an odd last column, every tile cut along k,
# the last round's
PAIRED = [(4100, 2047, 4104, 2), (2040, 2040, 8200, 1), (4001, 1000, 1032, 3), (2040, 2040, 1416, 1), (4001, 1000, 4200, 1), (2040, 2047, 4200, 1),
          (1016, 768, 5000, 1), (300, 2048, 8192, 1), (4096, 1024, 4096, 1)]


# shapes that the planner gives to 128 columns by 128, 160 or 192 rows in NN or NT (TN has none): the same edges, slices of the fewest
# rows, five partial stages to a tile (as short as they take), every tile and the last round's cut along k
NARROW = [(300, 16384, 40, 5), (4100, 2047, 1000, 3), (496, 2560, 520, 5), (300, 16376, 2056, 1), (1554, 2559, 1000, 3), (496, 8184, 2056, 1), (300, 4090, 12296, 1), (1554, 2560, 2560, 1)]
NARROW_NT = [(620, 6000, 4104, 3), (384, 12500, 4104, 3)]


@pytest.mark.parametrize("shape", SHAPES + PAIRED + NARROW, ids=str)
@pytest.mark.parametrize("layout", ["NN", "NT", "TN"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tiles_of_256_columns(layout, shape, dtype):
    _check(layout, shape, dtype)


# 128 x 128 tiles of one group with k-contiguous B, whole and in a sliced last round: long reductions over several steps alone
@pytest.mark.parametrize("shape", NARROW_NT, ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tiles_of_one_group_in_nt(shape, dtype):
    _check("NT", shape, dtype)


def _check(layout, shape, dtype):
    from cubework_amd import ops

    M, N, K, steps = shape
    pad = -N % 8  # B's rows are 16-byte aligned (an odd N has an odd output alone)
    a_shape, b_shape = ((K, M) if layout == "TN" else (M, K)), ((N, K) if layout == "NT" else (K, N + pad))
    A = [randn(a_shape, dtype, 3 * i).cuda() for i in range(steps)]
    B = [randn(b_shape, dtype, 3 * i + 1, std=0.05).cuda()[:, :K if layout == "NT" else N] for i in range(steps)]
    bias, add = randn((N,), dtype, 90).cuda(), randn((M, N + pad), dtype, 91).cuda()[:, :N]
    act = None if layout == "TN" else "relu"
    got = ops.gemm_ksteps(layout, A, B, bias, act, [add], want_preact=True)
    rows = torch.cat([torch.arange(0, min(M, 48)), torch.arange(max(M // 2 - 24, 0), M // 2 + 24), torch.arange(max(M - 48, 0), M)]).unique().cuda()
    want = add[rows].double() + bias.double()
    for a, b in zip(A, B):
        a64 = a[:, rows].double().t().contiguous() if layout == "TN" else a[rows].double()
        want += a64 @ (b.double().t().contiguous() if layout == "NT" else b.double())
    # fp32 sums rounded once: the storage type's bar
    assert_parity(got[1][rows], want, dtype, "preact %s %s %s" % (layout, shape, dtype))
    assert_parity(got[0][rows], want if act is None else want.clamp_min(0), dtype, "out %s %s %s" % (layout, shape, dtype))
    plain = ops.gemm_ksteps(layout, A, B)  # whole tiles' stores are counted, not waited for
    assert_parity(plain[rows], want - add[rows].double() - bias.double(), dtype, "plain %s %s %s" % (layout, shape, dtype))


@pytest.mark.parametrize("layout,M,N,K", [("NN", 300, 4096, 16384), ("NT", 1554, 2560, 7680), ("TN", 2040, 2296, 8200), ("NT", 4352, 4096, 1024),
                                          ("NN", 300, 2048, 8192), ("NT", 300, 4096, 12288), ("NT", 1552, 2560, 10240)])
def test_sliced_tiles(layout, M, N, K):
    """Every tile, or the last round's, cut along k; bias, addend and pre-activation behind the reduction."""
    from cubework_amd import _lib, ops

    a = randn((K, M) if layout == "TN" else (M, K), torch.bfloat16, 1).cuda()
    b = randn((N, K) if layout == "NT" else (K, N), torch.bfloat16, 2, 0.05).cuda()
    bias, add = randn((N,), torch.bfloat16, 3).cuda(), randn((M, N), torch.bfloat16, 4).cuda()
    assert _lib.load().cw_gemm_scratch_bytes(ops.LAYOUTS[layout], M, N, K, 1, a.stride(0), b.stride(0), 1, 1, 0, _lib.CW_BF16) > 0
    act = None if layout == "TN" else "gelu_tanh"
    out, pre = ops.gemm_ksteps(layout, [a], [b], bias, act, [add], want_preact=True)
    want = (a.double().t().contiguous() if layout == "TN" else a.double()) @ (b.double().t().contiguous() if layout == "NT" else b.double())
    want += bias.double() + add.double()
    assert_parity(pre, want, torch.bfloat16, "sliced preact")
    assert_parity(out, want if act is None else torch.nn.functional.gelu(want, approximate="tanh"), torch.bfloat16, "sliced out")


# K of every remainder by 8: the piece of 16 bytes in which a row ends, whole K inside a stage, steps and slices that end there; both
# sides of the planner's rule for long rows that are not whole lines
RAGGED_K = [(300, 50257, 37, 3), (300, 16384, 37, 5), (8184, 2040, 331, 3), (7000, 4600, 961, 1), (1023, 768, 12565, 1), (4001, 1000, 1039, 3), (4001, 1000, 4162, 1),
            (300, 16376, 2059, 1), (300, 4090, 12302, 1), (1554, 2560, 2556, 1), (300, 32768, 1021, 1),
            (4096, 1024, 12565, 1), (4096, 1024, 10235, 1)]


@pytest.mark.parametrize("shape", RAGGED_K, ids=str)
@pytest.mark.parametrize("layout", ["NN", "NT"])
def test_rows_that_end_inside_16_bytes(layout, shape):
    """What stands behind K in k-contiguous rows (NaN here) does not reach the sums."""
    from cubework_amd import ops

    M, N, K, steps = shape

    def rows_of_k(n, seed, std):
        t = torch.full((n, -(-K // 8) * 8), float("nan"), dtype=torch.bfloat16, device="cuda")
        t[:, :K] = randn((n, K), torch.bfloat16, seed, std).cuda()
        return t[:, :K]

    A = [rows_of_k(M, 3 * i, 1.0) for i in range(steps)]
    B = [rows_of_k(N, 3 * i + 1, 0.05) if layout == "NT" else randn((K, -(-N // 8) * 8), torch.bfloat16, 3 * i + 1, 0.05).cuda()[:, :N]
         for i in range(steps)]
    got = ops.gemm_ksteps(layout, A, B)
    rows = torch.cat([torch.arange(0, min(M, 64)), torch.arange(max(M - 64, 0), M)]).unique().cuda()
    want = sum(a[rows].double() @ (b.double().t().contiguous() if layout == "NT" else b.double()) for a, b in zip(A, B))
    assert_parity(got[rows], want, torch.bfloat16, "%s %s" % (layout, shape))
    assert bool(torch.isfinite(got).all())


# without addends rounded results go through LDS: tiles that lie whole in C and ones that don't (M, N, odd N), every height, sliced tiles;
# the bias absent, 16-byte aligned, 8-byte aligned, and neither; with and without the sums before the activation. Whole numbers: the sums
# are exact in fp32 (at most 9 K + 64 < 2^24), so every result is the exact one rounded once.
@pytest.mark.parametrize("shape", [(8192, 2048, 512), (8184, 2040, 328), (1552, 7672, 1352), (300, 32767, 1016), (7000, 4600, 1000), (4352, 4096, 1024)], ids=str)
@pytest.mark.parametrize("layout", ["NN", "NT", "TN"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_results_of_no_addends(layout, shape, dtype):
    from cubework_amd import ops

    M, N, K = shape
    gen = torch.Generator().manual_seed(M + N)
    whole = lambda *s: torch.randint(-3, 4, s, generator=gen).to(dtype).cuda()  # noqa: E731
    A = whole(*((K, M) if layout == "TN" else (M, K)))
    B = whole(N, K) if layout == "NT" else whole(K, N + -N % 8)[:, :N]
    sums = (A.t() if layout == "TN" else A).float() @ (B.t() if layout == "NT" else B).float()
    many = torch.randint(-64, 65, (N + 8,), generator=gen).to(dtype).cuda()
    for skip, act, preact in ((None, None, False), (0, None, False), (4, "relu", True), (1, "relu", False), (None, "relu", True), (0, "relu", True)):
        if layout == "TN" and act is not None:
            continue
        bias = None if skip is None else many[skip:skip + N]
        want = sums if bias is None else sums + bias.float()
        got = ops.gemm_ksteps(layout, [A], [B], bias, act, [], want_preact=preact)
        out, pre = got if preact else (got, None)
        assert torch.equal(out, (want if act is None else want.relu()).to(dtype)), (skip, act, preact)
        assert pre is None or torch.equal(pre, want.to(dtype)), (skip, act, preact)


# more than 16 slices: 256-column tiles of 256 and 224 rows, 128-column ones of 192, slices of unequal lengths, a ragged last k. Products of
# -1, 0 and 1, whose sums (at most K < 2^24) are exact in fp32 in any order.
@pytest.mark.parametrize("layout,M,N,K", [("NN", 1023, 768, 50257), ("TN", 1023, 768, 50257), ("NT", 1023, 768, 50257), ("NN", 403, 1280, 50304),
                                          ("NN", 178, 1536, 51072)])
def test_many_slices(layout, M, N, K):
    from cubework_amd import ops

    gen = torch.Generator().manual_seed(K)
    sign = lambda *s: torch.randint(-1, 2, s, generator=gen).bfloat16().cuda()  # noqa: E731
    rows8 = lambda r, c: sign(r, c + -c % 8)[:, :c]  # noqa: E731
    A = rows8(K, M) if layout == "TN" else rows8(M, K)
    B = rows8(N, K) if layout == "NT" else rows8(K, N)
    want = (A.t() if layout == "TN" else A).float() @ (B.t() if layout == "NT" else B).float()
    assert torch.equal(ops.gemm_ksteps(layout, [A], [B]), want.bfloat16())
