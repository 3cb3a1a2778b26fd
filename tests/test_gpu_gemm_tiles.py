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


# (K, N, rows): the planner gives 64 x 64, 128 x 128 (8 wavefronts), 192 x 128, 128 x 256 and 224 x 256 tiles to the rows of the first,
# 64 x 128, 128 x 128 (8 wavefronts) and 128 x 256 to those of the others (tests/test_gemm_plans.py): both matrix instructions, 32x32x16
# and 16x16x32, trips of 32 and of 64 k
ORDERED = [(2560, 7680, (64, 300, 600, 900, 1554)), (4096, 4096, (300, 600, 1600)), (2044, 4096, (300, 600, 1600))]


@pytest.mark.parametrize("K,N,rows", ORDERED)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_forward_rows_do_not_depend_on_the_kernel(K, N, rows, dtype):
    """The same across every kernel that a projection's row can meet: terms of very different size, so that sums in another order or
    through another rounding would show."""
    from cubework_amd import ops

    M = max(rows)
    a = (randn((M, K), torch.float32, 1) * torch.exp2(randn((M, K), torch.float32, 2))).to(dtype).cuda()
    b = randn((K, N), dtype, 3, 0.02).cuda()
    whole = ops.gemm_ksteps("NN", [a], [b])
    for r in rows:
        assert torch.equal(ops.gemm_ksteps("NN", [a[:r]], [b]), whole[:r])


def _abi_gemm(layout, A, B, bias, epilogue, scratch, addend=None):
    """cw_gemm_ksteps_ws as a C caller makes it, with `scratch` bytes of scratch."""
    import ctypes

    from cubework_amd import _lib
    from cubework_amd.ops import LAYOUTS, _dtype_code, _ld, _p, _ptr_table, _stream

    M, K = A.shape[::-1] if layout == "TN" else A.shape
    N = B.shape[0] if layout == "NT" else B.shape[1]
    C = torch.full((M, N), float("nan"), dtype=A.dtype, device=A.device)
    ws = torch.empty(max(scratch, 16), dtype=torch.uint8, device=A.device)
    add = [] if addend is None else [addend]
    rc = _lib.load().cw_gemm_ksteps_ws(LAYOUTS[layout], M, N, K, 1, _ptr_table([A]), _ld(A), _ptr_table([B]), _ld(B), _p(bias), epilogue, _p(C),
                                       _ld(C), ctypes.c_void_p(0), 0, _ptr_table(add), len(add), N, _p(ws) if scratch else None, scratch,
                                       _dtype_code(A), _stream())
    _lib.check(rc, "cw_gemm_ksteps_ws")
    return C


# whole tiles; every tile sliced (a long reduction over few tiles); unaligned rows without scratch for their copy (the
# register-staged kernel); the two fp32 kernels
@pytest.mark.parametrize("layout,M,N,K,dtype,pad,sliced", [
    ("NN", 300, 264, 64, torch.bfloat16, 0, False), ("NT", 64, 768, 3072, torch.float16, 0, True),
    ("NN", 130, 70, 50, torch.bfloat16, 3, False), ("NN", 130, 72, 40, torch.float32, 0, False),
    ("NN", 4096, 2048, 64, torch.float32, 0, False)])
def test_no_epilogue_ignores_a_bias_pointer(layout, M, N, K, dtype, pad, sliced):
    """CW_EPI_NONE is acc (+ addends) whatever the bias argument holds: the same bits as without a bias."""
    from cubework_amd import _lib
    from cubework_amd.ops import LAYOUTS, _dtype_code, _ld

    a = randn((M, K + pad), dtype, 1).cuda()[:, :K]
    b = randn((N, K + pad) if layout == "NT" else (K, N), dtype, 2, 0.05).cuda()[:, :K if layout == "NT" else N]
    bias, add = torch.full((N,), 1000.0, dtype=dtype, device="cuda"), randn((M, N), dtype, 3).cuda()
    scratch = 0 if pad else _lib.load().cw_gemm_scratch_bytes(LAYOUTS[layout], M, N, K, 1, _ld(a), _ld(b), 1, 1, 0, _dtype_code(a))
    assert (scratch > 0) == sliced
    for addend in (None, add):
        with_bias = _abi_gemm(layout, a, b, bias, _lib.CW_EPI_NONE, scratch, addend)
        assert torch.equal(with_bias, _abi_gemm(layout, a, b, None, _lib.CW_EPI_NONE, scratch, addend))
        want = a.double().cpu() @ (b.double().cpu().t() if layout == "NT" else b.double().cpu()) + (0 if addend is None else addend.double().cpu())
        assert_parity(with_bias, want, dtype, "no epilogue beside a bias pointer")


# Calls whose scratch is less than the best plan's: none, or cw_gemm_workspace_bytes
@pytest.mark.parametrize("layout,M,N,K,workspace", [
    ("NN", 256, 512, 8192, False),     # 128 x 128 tiles
    ("NT", 2600, 6160, 1024, False),   # 256 x 256 tiles
    ("NT", 4352, 4096, 1024, False),   # 256 x 256 tiles and a strip of 256 rows
    ("TN", 256, 256, 16384, True),     # 256 x 256 tiles in eight slices
    ("NT", 2600, 6160, 1032, False),   # the best plan without scratch
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_calls_with_less_scratch(layout, M, N, K, workspace, dtype):
    from cubework_amd import _lib
    from cubework_amd.ops import LAYOUTS, _dtype_code, _ld

    a = randn((K, M) if layout == "TN" else (M, K), dtype, 1)
    b = randn((N, K) if layout == "NT" else (K, N), dtype, 2, 0.05)
    bias, add = randn((N,), dtype, 3), randn((M, N), dtype, 4)
    lib, code = _lib.load(), LAYOUTS[layout]
    scratch = lib.cw_gemm_workspace_bytes(code, M, N, K, 1, _dtype_code(a)) if workspace else 0
    assert scratch < lib.cw_gemm_scratch_bytes(code, M, N, K, 1, _ld(a), _ld(b), 1, 1, 0, _dtype_code(a))
    assert (scratch > 0) == workspace
    got = _abi_gemm(layout, a.cuda(), b.cuda(), bias.cuda(), _lib.CW_EPI_BIAS, scratch, add.cuda())
    want = (a.float().t() if layout == "TN" else a.float()) @ (b.float().t() if layout == "NT" else b.float()) + bias.float() + add.float()
    assert_parity(got, want, dtype, "%s %dx%dx%d with %d bytes of scratch" % (layout, M, N, K, scratch))


@pytest.mark.parametrize("M,N,K,steps", [(1992, 2040, 4099, 1), (1992, 2040, 1030, 2), (2048, 2048, 8192, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_weight_gradient_of_one_block_per_unit(M, N, K, steps, dtype):
    """At most one block per compute unit: ragged tiles, a reduction that ends inside a trip, a seam of two steps."""
    import oracle
    from cubework_amd import ops

    A = [randn((K, M), dtype, 3 * i) for i in range(steps)]
    B = [randn((K, N), dtype, 3 * i + 1, std=0.05) for i in range(steps)]
    add = [randn((M, N), dtype, 91)]
    want = oracle.gemm_ksteps("TN", A, B, None, None, add)
    got = ops.gemm_ksteps("TN", [a.cuda() for a in A], [b.cuda() for b in B], None, None, [t.cuda() for t in add])
    assert_parity(got, want, dtype, "TN %dx%dx%d steps=%d" % (M, N, K, steps))
