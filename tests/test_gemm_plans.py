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


@pytest.mark.parametrize("layout,M,N,K", [("NT", 2394, 576, 1536), ("NT", 1894, 1024, 1024), ("NT", 1280, 1024, 1024), ("NN", 1777, 768, 768),
                                          ("NN", 473, 3072, 768), ("NN", 351, 3072, 1024)])
def test_short_products_of_one_round_take_64_x_128_tiles(plans, layout, M, N, K):
    """140 to 240 tiles of 64 x 128 are one round of the chip; as 64 x 64 they share its units in pairs (10 to 20 % slower)."""
    assert plans([(layout, M, N, K, 1)]) == [(3, 64, -(-M // 64) * -(-N // 128), 1, 0)]
