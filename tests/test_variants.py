"""Kernel variants on the host (csrc/variants.hpp): every shape's rules name
variants that are compiled, and a launch whose variant is not refuses instead of
leaving its buffers unwritten."""
import importlib.util
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "fherma-polynomial-cuda_amd" / "csrc"


@pytest.fixture(scope="module")
def variant_check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("variants") / "variant_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", str(CSRC), str(ROOT / "tests" / "variant_check.cpp"),
                    "-o", str(exe)], check=True)
    return lambda *args: subprocess.run([str(exe)] + [str(x) for x in args], check=True, capture_output=True,
                                        text=True, timeout=100).stdout


def test_every_shape_has_its_variants(variant_check):
    out = variant_check().split()
    assert out[0] == "ok" and int(out[1]) > 100000


@pytest.mark.parametrize("n,limbs,primes,kernel", [
    (128, 61, 127, "reconstruct_wide<32>"), (128, 63, 131, "reconstruct_waves"), (2048, 64, 133, "reconstruct_waves"),
    (2048, 65, 135, "reconstruct_wide<32>"), (4096, 64, 133, "reconstruct_wide<32>"),
    (2048, 124, 257, "reconstruct_wide<32>"), (2048, 125, 259, "reconstruct_wide<64>"),
    (2048, 128, 265, "reconstruct_waves"), (4096, 128, 265, "reconstruct_wide<64>"),
    (2048, 252, 521, "reconstruct_wide<64>"), (4096, 253, 523, "reconstruct_waves"),
])
def test_reconstruction_of_few_tiles(variant_check, n, limbs, primes, kernel):
    assert variant_check(n, limbs, primes).splitlines()[-1] == kernel


def test_gpu_cases_reach_the_gemm_tiles_they_name(variant_check, polymul):
    """tests/test_gpu_gemm_variants.py: each case's kernels, and together every
    variant of the two GEMMs."""
    spec = importlib.util.spec_from_file_location("gemm_variants", ROOT / "tests" / "test_gpu_gemm_variants.py")
    cases = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(cases)
    reached = set()
    for n, limbs, kernels in cases.CASES:
        with polymul.Plan(n, 32 * limbs, limbs, cases.case_modulus(limbs), device=False) as plan:
            taken = variant_check(n, limbs, len(plan.primes())).splitlines()
        assert set(kernels) <= set(taken), (n, limbs, taken)
        reached |= {k.split()[0] for k in kernels}
    assert reached == {"conversion_gemm<1>", "conversion_gemm<2>", "crt_gemm<1>", "crt_gemm<2>", "crt_small"}


def test_every_list_of_variants_is_checked():
    """Wherever the launch code expands a list of variants into `if`s, the
    function throws first when the shape's variant is not in the list."""
    text = (CSRC / "kernels.hip").read_text()
    for launcher, check in (("launch_convert", "convert_compiled"), ("launch_ntt_rows_product", "rows_compiled"),
                            ("launch_ntt_forward_columns", "columns_compiled"),
                            ("launch_ntt_inverse_columns", "columns_compiled"),
                            ("launch_group", "convert_group_compiled")):
        body = text[text.index("\nvoid %s(" % launcher):]
        body = body[:body.index("\n}\n")]
        first = body.index("hipLaunchKernelGGL")
        assert re.search(r"if \([^;]*!%s\([^;]*throw std::logic_error" % check, body[:first]), launcher
