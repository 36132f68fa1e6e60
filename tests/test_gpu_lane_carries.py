"""Carries between the lanes of a coefficient in the reconstructions that give
it several lanes: the lane of word L + 1 ends the chain, wherever in its four
words that is, and the lanes above it stay out.  Limb counts on both sides of
each lane's edge and of each lane count (4, 8, 16, 32 and 64 lanes), through a
plan's own kernels (fused, or more than 8 tiles and up to 8) and a batch's, with a q of all
ones, a power of two, one limb of many, and random, and operands that make the
quotient estimate miss (q-1, zero).  Bit-exact, so there is no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMBS = [2, 3, 4, 10, 11, 14, 15, 27, 30, 31, 59, 63, 64, 95, 122, 123, 124, 126, 127, 128, 131, 250, 251, 252]


def _moduli(limbs, workloads, rng):
    power = np.zeros(limbs, dtype=np.uint32)
    power[-1] = 0x80000000
    short = np.zeros(limbs, dtype=np.uint32)
    short[0] = 0xFFFFFFFB
    return {"random": workloads.random_modulus(limbs, rng), "ones": np.full(limbs, 0xFFFFFFFF, dtype=np.uint32),
            "power": power, "short": short}


# up to 8 tiles: a wave per coefficient at 63, 64, 127, 128, 191 and 192 limbs only
FEW = [(n, limbs) for n in (128, 2048) for limbs in (62, 63, 64, 65, 126, 127, 128, 129, 190, 191, 192, 193)]


@pytest.mark.parametrize("n,limbs", [(4096 if limbs > 60 else 256, limbs) for limbs in LIMBS] + FEW)
def test_lane_ends(polymul, workloads, oracle, device_memory, n, limbs):
    print("[gpu-case] lane carries", n, limbs, flush=True)
    rng = np.random.default_rng(97000 + limbs)
    for kind, q in _moduli(limbs, workloads, rng).items():
        used = max(i + 1 for i in range(limbs) if q[i])
        a, b = (np.zeros((n, limbs), dtype=np.uint32) for _ in range(2))
        a[:, :used] = workloads.uniform_below(q[:used], n, rng)
        b[:, :used] = workloads.uniform_below(q[:used], n, rng)
        a[: n // 4] = workloads.q_minus_one(q)
        b[n // 2:] = 0
        b[0] = workloads.q_minus_one(q)
        expect = oracle.kronecker_gmp(a, b, q)
        with polymul.Plan(n, 32 * limbs, limbs, q) as plan:
            pa, pb, pc = (device_memory.upload(x) for x in (a, b, np.full_like(a, 0xDEADBEEF)))
            try:
                plan.multiply_device(pa, pb, pc)
                assert np.array_equal(device_memory.download(pc, a.shape, np.uint32), expect), "%s q" % kind
                device_memory.write(pc, np.full_like(a, 0xDEADBEEF))
                polymul.multiply_device_batch([plan], [pa], [pb], [pc])
                assert np.array_equal(device_memory.download(pc, a.shape, np.uint32), expect), "%s q, batch" % kind
            finally:
                for ptr in (pa, pb, pc):
                    device_memory.free(ptr)


def test_narrower_q_is_not_slower(polymul, workloads, device_memory):
    """q of 128 limbs leaves 31 of a coefficient's 64 lanes empty.  Its
    reconstruction may not take longer than that of 252 limbs, which fills
    them all and has twice the words (kernel times, the shortest of 30; 1.5
    times as long is allowed for the clock)."""
    print("[gpu-case] reconstruction of 128 and 252 limbs", flush=True)
    n, best = 4096, {}
    rng = np.random.default_rng(98000)
    for limbs in (252, 128):
        q = workloads.random_modulus(limbs, rng)
        a, b = workloads.uniform_below(q, n, rng), workloads.uniform_below(q, n, rng)
        with polymul.Plan(n, 32 * limbs, limbs, q) as plan:
            pa, pb, pc = (device_memory.upload(x) for x in (a, b, a))
            try:
                plan.set_profiling(True)
                times = []
                for _ in range(30):
                    plan.multiply_device(pa, pb, pc)
                    times.append(plan.stage_times()["reconstruct"])
            finally:
                for ptr in (pa, pb, pc):
                    device_memory.free(ptr)
        best[limbs] = min(times)
    print("[gpu-case] us:", {limbs: round(1000 * t, 1) for limbs, t in best.items()}, flush=True)
    assert best[128] < 1.5 * best[252]
