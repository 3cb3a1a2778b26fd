"""GPU parity of the bias-gradient column sum and the fused-activation
backward (through the C ABI) against the CPU oracle."""
import pytest
import torch

from tests.util import assert_parity, randn

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
SHAPES = [(8192, 2048), (100, 1000), (33, 8), (5, 7), (1000, 520), (4096, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_colsum(shape, dtype):
    import oracle
    from cubework_amd import ops

    M, N = shape
    dy = randn((M, N), dtype, 1)
    got = ops.colsum(dy.to(DEV))
    with oracle.precision(torch.float64):
        want = oracle.colsum(dy)
    # a sum of M terms per column, against its float64 value
    assert_parity(got, want, torch.float32, "colsum")
    # determinism: two runs are bit identical
    assert torch.equal(got, ops.colsum(dy.to(DEV)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("act", [None, "gelu_tanh", "gelu_erf", "relu"])
@pytest.mark.parametrize("shape", [(1024, 512), (77, 130), (9, 5)])
def test_act_bwd_colsum(shape, act, dtype):
    import oracle
    from cubework_amd import ops

    M, N = shape
    dy = randn((M, N), dtype, 2)
    pre = randn((M, N), dtype, 3, std=1.5)
    dpre, dbias = ops.act_bwd_colsum(act, dy.to(DEV), pre.to(DEV))
    with oracle.precision(torch.float64):
        want_dpre, want_dbias = oracle.act_bwd_colsum(act, dy, pre)
    assert_parity(dpre, want_dpre, dtype, "dPre")
    assert_parity(dbias, want_dbias, torch.float32, "dbias")
    dpre2, none = ops.act_bwd_colsum(act, dy.to(DEV), pre.to(DEV), want_dbias=False)
    assert none is None and torch.equal(dpre, dpre2)


def test_colsum_padded_rows():
    import oracle
    from cubework_amd import ops

    parent = randn((300, 136), torch.bfloat16, 4).to(DEV)
    view = parent[:, :128]
    with oracle.precision(torch.float64):
        want = oracle.colsum(view.cpu())
    assert_parity(ops.colsum(view), want, torch.float32, "padded colsum")


def test_mfma_rate_diagnostic_runs_in_every_mode():
    """cw_diag_mfma_rate (the measurement aid behind bench.py's MFMA ceilings, in the measurement library): zero
    operands leave zero sums; random operands, from registers or read from LDS, leave finite non-zero ones, the
    same on every call."""
    from cubework_amd import _diag

    lib = _diag.load()
    sink = torch.full((65536,), float("nan"), dtype=torch.float32, device=DEV)
    assert lib.cw_diag_mfma_rate(3, 1, sink.data_ptr(), None) == 0
    torch.cuda.synchronize()
    assert torch.equal(sink, torch.zeros_like(sink))
    for mode in (0, 2):
        runs = []
        for _ in range(2):
            sink.fill_(float("nan"))
            assert lib.cw_diag_mfma_rate(4, mode, sink.data_ptr(), None) == 0
            torch.cuda.synchronize()
            runs.append(sink.clone())
        assert torch.isfinite(runs[0]).all() and (runs[0] != 0).any()
        assert torch.equal(runs[0], runs[1])


def test_gemm_part_diagnostic_whole_kernel_matches_the_library():
    """cw_diag_gemm_part with part 0 is the library's launch for the benchmark's shape: bit-equal to cw_gemm_ksteps; parts 1 to 3
    (4 wavefronts; no operand loads / no epilogue / no LDS reads in the k loop) run and return."""
    import ctypes
    from cubework_amd import _diag, ops

    lib = _diag.load()
    M, N, K = 8192, 2048, 512   # 256 tiles: the shape class the library gives to this kernel
    A = [randn((M, K), torch.bfloat16, 40 + i).to(DEV) for i in range(2)]
    B = [randn((K, N), torch.bfloat16, 50 + i, 0.05).to(DEV) for i in range(2)]
    bias = randn((N,), torch.bfloat16, 60, 0.1).to(DEV)
    want = ops.gemm_ksteps("NN", A, B, bias, "gelu_tanh")
    ta = (ctypes.c_void_p * 2)(*[t.data_ptr() for t in A])
    tb = (ctypes.c_void_p * 2)(*[t.data_ptr() for t in B])
    out = torch.empty_like(want)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.cw_diag_gemm_part(0, M, N, K, 2, ta, K, tb, N, bias.data_ptr(), out.data_ptr(), N, stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    for part in (1, 2, 3):
        assert lib.cw_diag_gemm_part(part, M, N, K, 2, ta, K, tb, N, bias.data_ptr(), out.data_ptr(), N, stream) == 0
    torch.cuda.synchronize()


@pytest.mark.parametrize("steps", [1, 2])
def test_gemm_part_diagnostic_takes_k_of_128(steps):
    """cw_diag_gemm_part's shortest K: two stages of 64 k (one step), fewer than the library's 256 x 256 kernel takes, and four."""
    import ctypes
    from cubework_amd import _diag

    lib = _diag.load()
    M, N, K = 4096, 2048, 128
    A = [randn((M, K), torch.bfloat16, 40 + i).to(DEV) for i in range(steps)]
    B = [randn((K, N), torch.bfloat16, 50 + i, 0.05).to(DEV) for i in range(steps)]
    bias = randn((N,), torch.bfloat16, 60, 0.1).to(DEV)
    ta = (ctypes.c_void_p * steps)(*[t.data_ptr() for t in A])
    tb = (ctypes.c_void_p * steps)(*[t.data_ptr() for t in B])
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    want = torch.nn.functional.gelu(sum(a.double() @ b.double() for a, b in zip(A, B)) + bias.double(), approximate="tanh")
    for part in (0, 4):
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert lib.cw_diag_gemm_part(part, M, N, K, steps, ta, K, tb, N, bias.data_ptr(), out.data_ptr(), N, stream) == 0
        assert_parity(out, want, torch.bfloat16, "part %d, %d steps of 128" % (part, steps))
    for part in (1, 2, 3):
        assert lib.cw_diag_gemm_part(part, M, N, K, steps, ta, K, tb, N, bias.data_ptr(), out.data_ptr(), N, stream) == 0
    torch.cuda.synchronize()


@pytest.mark.parametrize("M", [1, 3, 63, 64, 65, 160, 161, 224, 225, 255, 256, 257, 511, 512, 513])  # the last rows of the one-launch kernels among them
@pytest.mark.parametrize("N", [8, 120, 136, 1000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_column_sums_of_few_rows(M, N, dtype):
    """One launch up to 512 rows (256 with an activation in fp32, 224 in 16 bits, 160 of a GELU), NaN outside the operands' columns; fp32 sums of M values in any order lie
    within M 2^-24 of the sum of magnitudes. dPre does not depend on the kernel."""
    from cubework_amd import ops

    def place(t):
        buf = torch.full((M + 1, N + 16), float("nan"), dtype=dtype, device=DEV)
        buf[:M, :N] = t
        return buf[:M, :N]

    dy, pre = (place(randn((M, N), dtype, 7 * M + k, device=DEV)) for k in range(2))
    for out in (torch.float32, dtype):
        got = ops.colsum(dy, out_dtype=out)
        want, room = dy.double().sum(0), dy.double().abs().sum(0) * M * 2.0 ** -24
        room = room + want.abs() * (0 if out == torch.float32 else torch.finfo(out).eps / 2) * 1.001
        assert got.dtype == out and (got.double() - want).abs().le(room).all()
    for act in ("gelu_tanh", "gelu_erf", "relu"):
        dpre, db = ops.act_bwd_colsum(act, dy, pre)
        alone, none = ops.act_bwd_colsum(act, dy, pre, want_dbias=False)
        assert none is None and torch.equal(dpre, alone)
        # the sums are of the unrounded products: 16-bit rounding of each on top where dPre is 16 bits
        per = 2.0 ** -24 * M + (0 if dtype == torch.float32 else torch.finfo(dtype).eps / 2)
        assert (db.double() - dpre.double().sum(0)).abs().le(dpre.double().abs().sum(0) * per * 1.01 + 1e-6).all()


@pytest.mark.parametrize("M", [1, 256, 257, 512, 513])
def test_column_sums_refuse_scratch_that_is_too_small_at_every_size(M):
    """Less than one row of partial sums, also where the launch needs none: refused before anything is written."""
    import ctypes

    from cubework_amd import _lib

    N, lib = 64, _lib.load()
    dy, pre = (randn((M, N), torch.bfloat16, k, device=DEV) for k in range(2))
    dpre, out = torch.zeros_like(dy), torch.zeros(N, device=DEV)
    need = lib.cw_colsum_workspace_bytes(M, N)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for size, rc in ((N * 4 - 1, _lib.CW_ERR_INVALID), (need, 0)):
        assert lib.cw_colsum(M, N, p(dy), N, p(out), 1, p(ws), size, 0, stream) == rc
        assert lib.cw_act_bwd_colsum(2, M, N, p(dy), N, p(pre), N, p(dpre), N, p(out), 1, p(ws), size, 0, stream) == rc
        assert out.any().item() == dpre.any().item() == (rc == 0)
