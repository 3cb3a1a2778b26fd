"""Which tiles the planner of the 16-bit block GEMM (cubework_amd/csrc/gemm_plan.hip) gives to products, on the CPU: rules that a
change of its cost model must not lose."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cubework_amd", "csrc")
LAYOUTS = {"NN": 0, "NT": 1, "TN": 2}
PAIRED = 5  # configuration: 128 x 128 tiles with two groups of wavefronts along k


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    """[(layout, M, N, K, steps)] -> [(cfg, rows, full, slices, rest)], operands in rows of a multiple of 8."""
    hipcc = next((c for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")) if c and os.path.exists(c)), None)
    if hipcc is None:
        pytest.skip("hipcc not found")
    exe = str(tmp_path_factory.mktemp("plans") / "plan_print")
    build = subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            "-Wno-unused-command-line-argument", os.path.join(ROOT, "tests", "host", "plan_print.hip"),
                            os.path.join(CSRC, "gemm_plan.hip"), os.path.join(CSRC, "cw_runtime.hip"), "-o", exe],
                           capture_output=True, text=True, timeout=600)
    assert build.returncode == 0, build.stdout + build.stderr

    def plan(products):
        lines = ["%d %d %d %d %d %d %d 1 1" % (LAYOUTS[lay], M, N, K, steps, -(-(M if lay == "TN" else K) // 8) * 8, -(-(K if lay == "NT" else N) // 8) * 8)
                 for lay, M, N, K, steps in products]
        run = subprocess.run([exe], input="\n".join(lines), capture_output=True, text=True, timeout=60)
        assert run.returncode == 0, run.stderr
        return [tuple(int(v) for v in line.split()) for line in run.stdout.splitlines()]
    return plan


@pytest.mark.parametrize("layout,M,N,K", [("NN", 251, 2048, 50272), ("NN", 2048, 1024, 12568), ("NN", 1632, 768, 12568)])
def test_long_rows_in_short_blocks_stay_on_the_paired_kernel(plans, layout, M, N, K):
    """Rows that are not whole 128-byte lines slow the paired kernel by the length of a block's walk, not of the product's."""
    (cfg, _, full, slices, _), = plans([(layout, M, N, K, 1)])
    assert (cfg, full) == (PAIRED, 0) and -(-K // 128) / slices <= 80


def test_long_rows_in_long_blocks_leave_the_paired_kernel(plans):
    (cfg, *_), = plans([("NN", 4096, 1024, 12568, 1)])
    assert cfg != PAIRED


@pytest.mark.parametrize("M,N,K", [(1554, 768, 2304), (489, 2560, 2560), (2561, 768, 3072)])
def test_input_gradients_of_one_round_take_64_x_128_tiles(plans, M, N, K):
    """At most 256 tiles of 64 x 128, whose operands move as whole lines: 17 to 23 % faster than slices of the paired kernel's."""
    assert plans([("NT", M, N, K, 1)]) == [(3, 64, -(-M // 64) * -(-N // 128), 1, 0)]


@pytest.mark.parametrize("M,N,K", [(58, 876, 3712), (49, 896, 2752), (185, 768, 2304)])
def test_few_rows_are_not_cut_into_more_slices_than_pay(plans, M, N, K):
    """Every slice is a wait of the reduction: 4 to 6 are 11 to 18 % faster than the 7 to 15 that fill the chip."""
    (cfg, _, full, slices, _), = plans([("NT", M, N, K, 1)])
    assert (cfg, full) == (4, 0) and 3 <= slices <= 6


@pytest.mark.parametrize("layout,M,N,K", [("NT", 2394, 576, 1536), ("NT", 1894, 1024, 1024), ("NT", 1280, 1024, 1024), ("NN", 1777, 768, 768),
                                          ("NN", 473, 3072, 768), ("NN", 351, 3072, 1024)])
def test_short_products_of_one_round_take_64_x_128_tiles(plans, layout, M, N, K):
    """140 to 240 tiles of 64 x 128 are one round of the chip; as 64 x 64 they share its units in pairs (10 to 20 % slower)."""
    assert plans([(layout, M, N, K, 1)]) == [(3, 64, -(-M // 64) * -(-N // 128), 1, 0)]


@pytest.mark.parametrize("layout,M,N,K", [("NN", 1023, 768, 50257), ("TN", 1023, 768, 50257), ("NT", 1023, 768, 50257), ("NN", 403, 1280, 50304)])
def test_few_large_tiles_of_a_long_k_fill_the_chip(plans, layout, M, N, K):
    """Sixteen slices of 10 or 12 tiles of 256 x 256 would leave a third of the units idle, and the paired kernel was chosen (up to 40 % slower)."""
    (cfg, _, full, slices, rest), = plans([(layout, M, N, K, 1)])
    assert (cfg, full) == (0, 0) and slices > 16 and slices * rest <= 256


@pytest.mark.parametrize("M,N,K", [(34, 3072, 56535), (68, 2048, 50304), (128, 2048, 50257)])
def test_few_rows_are_left_to_the_small_tiles(plans, M, N, K):
    (cfg, _, _, slices, _), = plans([("TN", M, N, K, 1)])
    assert cfg != 0 and slices <= 16


@pytest.mark.parametrize("M,N,K", [(768, 3072, 4416), (3072, 768, 5295), (3072, 768, 6528), (1024, 3072, 6080)])
def test_weight_gradients_are_not_cut_into_many_slices_of_large_tiles(plans, M, N, K):
    """Six or seven slices of 36 tiles of 256 x 256 took 20 % longer than three of 128 x 256 or whole 128 x 128 tiles."""
    (cfg, _, full, slices, _), = plans([("TN", M, N, K, 1)])
    assert cfg != 0 or full > 0 or slices <= 3


@pytest.mark.parametrize("M,N,K,cfg", [(50257, 1024, 166, 1), (50272, 2048, 188, 1), (50272, 1024, 250, 1), (50257, 2560, 250, 0)])
def test_vocabulary_gradients_of_few_tokens(plans, M, N, K, cfg):
    """Four stages of k: 256 x 256 tiles only where their last round is fuller than a quarter."""
    assert plans([("TN", M, N, K, 1)])[0][0] == cfg


@pytest.mark.parametrize("layout,M,N,K", [("TN", 2820, 1632, 166), ("TN", 3520, 1664, 407), ("NT", 6243, 832, 256), ("NN", 6620, 544, 288)])
def test_short_products_of_half_a_round_take_128_x_128_tiles(plans, layout, M, N, K):
    """160 to 200 tiles of 128 x 256 would leave each of its blocks alone on its unit (15 to 25 % slower)."""
    assert plans([(layout, M, N, K, 1)])[0][:2] == (2, 128)


@pytest.mark.parametrize("M,N,K,cfg", [(7948, 2560, 2560, 1), (2465, 7680, 2560, 1), (2028, 10240, 2560, 1), (14502, 2560, 2560, 0), (1554, 10240, 2560, 6)])
def test_forward_products_of_many_rounds_take_256_columns(plans, M, N, K, cfg):
    """More than two and a half rounds of 128-column tiles are slower than the larger ones' (7 to 15 %)."""
    assert plans([("NN", M, N, K, 1)])[0][0] == cfg


# What the lists of the GPU tests are there for: configuration, tile height, and w (whole tiles), s (every tile cut along k) or m (the
# last round's cut), in NN, NT and TN. A plan that moves takes a kernel's coverage with it: find the list another shape then.
WIDE_PLANS = {
    "SHAPES": {(300, 50257, 40, 3): "0x160w 0x160w 0x160w", (4100, 4090, 392, 1): "1x128w 0x256m 0x256m", (300, 32768, 1016, 1): "0x160w 0x160w 0x160w",
               (376, 32760, 1000, 1): "0x192w 0x192w 0x192w", (1552, 7672, 1352, 1): "0x224w 0x224w 0x224w",
               (8184, 2040, 328, 3): "0x256w 0x256w 1x128w", (8184, 6136, 520, 1): "0x256w 0x256w 0x256w",
               (7000, 4600, 1000, 1): "0x256w 0x256w 0x256w", (1024, 25003, 768, 1): "0x256w 0x256w 0x256w", (8192, 2048, 512, 2): "0x256w 0x256w 0x256w"},
    "PAIRED": {(4100, 2047, 4104, 2): "5x128m 5x128m 5x128m", (2040, 2040, 8200, 1): "5x128w 5x128w 5x128w",
               (4001, 1000, 1032, 3): "5x128w 5x128w 5x128w", (2040, 2040, 1416, 1): "2x128w 5x128w 2x128w",
               (4001, 1000, 4200, 1): "5x128w 5x128w 5x128w", (2040, 2047, 4200, 1): "5x128w 5x128w 5x128w",
               (1016, 768, 5000, 1): "5x128s 5x128s 4x64w", (300, 2048, 8192, 1): "5x128s 5x128s 5x128s", (4096, 1024, 4096, 1): "5x128w 5x128w 5x128w"},
    "NARROW": {(300, 16384, 40, 5): "6x160w 6x160w 2x128w", (4100, 2047, 1000, 3): "6x192w 6x192m 5x128m", (496, 2560, 520, 5): "3x64w 7x128s 3x64w",
               (300, 16376, 2056, 1): "6x160w 6x160w 0x160s", (1554, 2559, 1000, 3): "6x192w 6x192w 3x64w",
               (496, 8184, 2056, 1): "7x128w 5x128w 5x128w", (300, 4090, 12296, 1): "6x160s 6x160s 0x160s", (1554, 2560, 2560, 1): "6x192w 6x192w 3x64w"},
    "RAGGED_K": {(300, 50257, 37, 3): "0x160w 0x160w", (300, 16384, 37, 5): "6x160w 6x160w", (8184, 2040, 331, 3): "0x256w 0x256w",
                 (7000, 4600, 961, 1): "0x256w 0x256w", (1023, 768, 12565, 1): "5x128s 5x128s", (4001, 1000, 1039, 3): "5x128w 5x128w",
                 (4001, 1000, 4162, 1): "5x128w 5x128w", (300, 16376, 2059, 1): "6x160w 6x160w", (300, 4090, 12302, 1): "6x160s 6x160s",
                 (1554, 2560, 2556, 1): "6x192w 6x192w", (300, 32768, 1021, 1): "0x160w 0x160w", (4096, 1024, 12565, 1): "0x256s 0x256s",
                 (4096, 1024, 10235, 1): "5x128w 5x128w"},
}


def _code(plan):
    cfg, rows, full, _, rest = plan
    return "%dx%d%s" % (cfg, rows, "w" if rest == 0 else "s" if full == 0 else "m")


@pytest.mark.parametrize("name", sorted(WIDE_PLANS))
def test_the_gpu_tests_reach_the_kernels_they_name(plans, name):
    from tests import test_gpu_gemm_wide as gpu

    shapes = getattr(gpu, name)
    assert sorted(WIDE_PLANS[name]) == sorted(shapes)
    for shape in shapes:
        want = WIDE_PLANS[name][shape].split()
        assert [_code(p) for p in plans([(lay, *shape) for lay in ("NN", "NT", "TN")[:len(want)]])] == want, shape


def test_the_gpu_tests_reach_the_kernels_they_compare(plans):
    from tests import test_gpu_gemm_tiles as tiles
    from tests import test_gpu_gemm_wide as wide

    assert [_code(p) for p in plans([("NT", *s) for s in wide.NARROW_NT])] == ["7x128w", "7x128m"]
    ordered = [[_code(p) for p in plans([("NN", m, N, K, 1) for m in rows])] for K, N, rows in tiles.ORDERED]
    assert ordered == [["4x64w", "7x128w", "6x160w", "1x128w", "0x224w"], ["3x64w", "7x128w", "1x128w"], ["3x64w", "7x128w", "1x128w"]]
