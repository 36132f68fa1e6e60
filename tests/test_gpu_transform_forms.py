"""The transforms' lazy forms against the oracle where their ranges are tight:
every row width of the register row kernel (128 to 2048; 64 takes the LDS one)
and row count of the register column kernels (2 to 64), each base case (n1 =
1, 2, 4, 8, whose last level hands different ranges on) and primes just below
2^31, with operands that are all q-1, alternate 0 and q-1, and random.
Bit-exact, so there is no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 128, 256, 512, 1024, 2048, 4096, 8192, 16384, 32768, 65536, 131072])
@pytest.mark.parametrize("block", [1, 2, 4, 8])
def test_forms(polymul, workloads, oracle, n, block):
    print("[gpu-case] transform forms", n, block, flush=True)
    limbs = 2
    rng = np.random.default_rng(94000 + n + block)
    q = workloads.random_modulus(limbs, rng)
    m = np.tile(workloads.q_minus_one(q), (n, 1))
    alt = m.copy()
    alt[::2] = 0
    a, b = workloads.uniform_below(q, n, rng), workloads.uniform_below(q, n, rng)
    with polymul.Plan(n, 32 * limbs, limbs, q, min_block=block) as plan:
        assert plan.info()["block"] == block
        for x, y in ((a, b), (m, m), (alt, m), (alt, b)):
            assert np.array_equal(plan.multiply(x, y), oracle.kronecker_gmp(x, y, q))
