"""The reconstructions with several lanes per coefficient against the oracle, at
the edges of their variants.  The kernel that does the CRT GEMM too: 12, 28 and
60 limbs are the widest q of one, two and four waves of word sums, 61 the
narrowest that takes the separate kernels; of those, 124 and 252 limbs are the
widest q of 32 and 64 lanes.  N below, at and above the blocks' coefficients,
enough of them for the separate kernels, and two, four and eight transform rows,
whose inverse column stages the fused kernel does; q all ones, a power of two, one,
and with zero limbs on top; operands random, all q-1 and zero.  Bit-exact, so
there is no tolerance."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _moduli(limbs, workloads, rng):
    ones = np.full(limbs, 0xFFFFFFFF, dtype=np.uint32)
    power = np.zeros(limbs, dtype=np.uint32)
    power[-1] = 0x80000000
    short = np.zeros(limbs, dtype=np.uint32)  # a one-limb q stored in `limbs` limbs
    short[0] = 0xFFFFFFFB
    return {"random": workloads.random_modulus(limbs, rng), "ones": ones, "power": power, "short": short}


LIMBS = [1, 2, 6, 12, 13, 28, 29, 60, 61, 62, 63, 124, 125, 251, 252, 253]


@pytest.mark.parametrize("n,limbs", [(n, limbs) for n in (1, 32, 64, 128, 1024) for limbs in LIMBS] +
                         [(4096, limbs) for limbs in LIMBS if limbs > 60] +
                         [(n, limbs) for n in (4096, 8192, 16384) for limbs in (12, 28, 60)])
def test_fused_reconstruction(polymul, workloads, oracle, n, limbs):
    rng = np.random.default_rng(91000 + 100 * limbs + n)
    for kind, q in _moduli(limbs, workloads, rng).items():
        print("[gpu-case] fused", n, limbs, kind, flush=True)
        sys.stdout.flush()
        used = max(i + 1 for i in range(limbs) if q[i])
        a = np.zeros((n, limbs), dtype=np.uint32)
        b = np.zeros((n, limbs), dtype=np.uint32)
        a[:, :used] = workloads.uniform_below(q[:used], n, rng)
        b[:, :used] = workloads.uniform_below(q[:used], n, rng)
        m = np.tile(workloads.q_minus_one(q), (n, 1))
        with polymul.Plan(n, 32 * limbs, limbs, q) as plan:
            for x, y in ((a, b), (m, m), (a, m), (np.zeros_like(a), b)):
                c = plan.multiply(x, y)
                assert np.array_equal(c, oracle.kronecker_gmp(x, y, q)), "%s q, N=%d, L=%d" % (kind, n, limbs)
