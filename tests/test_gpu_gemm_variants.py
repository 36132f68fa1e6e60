"""Each block tile of the two GEMMs against the oracle, through the device entry,
whose launches take all coefficients at once: every case names the kernels it is
there for, as the rules pick them from its N, limbs and primes (test_variants.py
checks the names on the host).  Halves in one short round and after a full one,
whole tiles in a full round, after two of them and with a short last one, and the
kernel that splits K over its waves with 8 to 17 K steps, which are all the
remainders of its two-deep loop.  Bit-exact, so there is no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# N, limbs, kernels (the number after a GEMM's name is its whole tiles, after crt_small's its K steps)
CASES = [
    (1024, 257, ["conversion_gemm<1> 72", "crt_small 34"]),
    (2048, 300, ["conversion_gemm<2> 160"]),
    (4096, 330, ["conversion_gemm<1> 352", "crt_gemm<1> 96"]),
    (8192, 300, ["conversion_gemm<2> 640", "crt_gemm<2> 160"]),
    (8192, 226, ["crt_gemm<1> 128"]),
    (16384, 226, ["crt_gemm<2> 256"]),
    (16384, 300, ["conversion_gemm<2> 1280", "crt_gemm<1> 320"]),
    (4096, 868, ["conversion_gemm<2> 928", "crt_gemm<2> 224"]),
    (32768, 226, ["crt_gemm<2> 512"]),
    (64, 61, ["crt_small 8"]), (64, 64, ["crt_small 9"]), (128, 72, ["crt_small 10"]), (256, 80, ["crt_small 11"]),
    (256, 90, ["crt_small 12"]), (512, 97, ["crt_small 13"]), (64, 105, ["crt_small 14"]), (256, 113, ["crt_small 15"]),
    (512, 120, ["crt_small 16"]), (256, 125, ["crt_small 17"]),
]


def case_modulus(limbs):
    """A modulus that any draw of operands may use: all ones but the lowest bits."""
    q = np.full(limbs, 0xFFFFFFFF, dtype=np.uint32)
    q[0] -= 4
    return q


@pytest.mark.parametrize("n,limbs", [case[:2] for case in CASES])
def test_gemm_variant(polymul, workloads, oracle, device_memory, n, limbs):
    print("[gpu-case] gemm variant", n, limbs, flush=True)
    rng = np.random.default_rng(96000 + n + limbs)
    q = case_modulus(limbs)
    a, b = workloads.uniform_below(q, n, rng), workloads.uniform_below(q, n, rng)
    a[0] = b[-1] = workloads.q_minus_one(q)
    expect = oracle.kronecker_gmp(a, b, q)
    with polymul.Plan(n, 32 * limbs, limbs, q) as plan:
        ptrs = [device_memory.upload(x) for x in (a, b, np.full_like(a, 0xDEADBEEF))]
        try:
            plan.multiply_device(*ptrs)
            assert np.array_equal(device_memory.download(ptrs[2], a.shape, np.uint32), expect)
        finally:
            for ptr in ptrs:
                device_memory.free(ptr)
