"""The GEMMs' block tiles against the oracle, with the sizes that pick each of
them: whole tiles, halves (few blocks, or a short last round) and, for the CRT
GEMM, 64 x 64 tiles whose waves split K (also fewer K steps than waves and every
remainder).  Bit-exact, so there is no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,limbs", [
    (1, 61), (64, 64), (256, 65),      # one tile, K steps 9 to 10
    (512, 70), (512, 80), (512, 100),  # the remainders of four K steps
    (2048, 129), (2048, 300),          # conversion GEMM in halves
    (4096, 226), (8192, 226),          # CRT GEMM in halves
    (16384, 226), (1024, 900),         # whole tiles
])
def test_tiles(polymul, workloads, oracle, n, limbs):
    print("[gpu-case] gemm tiles", n, limbs, flush=True)
    rng = np.random.default_rng(95000 + n + limbs)
    q = workloads.random_modulus(limbs, rng)
    a, b = workloads.uniform_below(q, n, rng), workloads.uniform_below(q, n, rng)
    a[0] = workloads.q_minus_one(q)
    with polymul.Plan(n, 32 * limbs, limbs, q) as plan:
        assert np.array_equal(plan.multiply(a, b), oracle.kronecker_gmp(a, b, q))
