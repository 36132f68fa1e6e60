"""The conversion that reads the limbs itself (q of up to 256 limbs) against the
oracle: residues exactly, for limb counts at the edges of its 64-byte K steps
and of its range, N below, at and above a block, and prime counts of one, two
and more 16-prime wave rows; then whole products, with enough coefficients for
its wider blocks, with one operand resident, and from device operands that
are only 4-byte aligned.  Bit-exact, so there is no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(workloads, n, limbs, seed):
    rng = np.random.default_rng(seed)
    q = workloads.random_modulus(limbs, rng)
    return q, workloads.uniform_below(q, n, rng), workloads.uniform_below(q, n, rng)


@pytest.mark.parametrize("limbs", [1, 2, 7, 8, 15, 16, 17, 32, 33, 64, 127, 128, 129, 255, 256, 257])
@pytest.mark.parametrize("n", [1, 64, 256])
def test_residues(polymul, workloads, oracle, n, limbs):
    print("[gpu-case] short conversion residues", n, limbs, flush=True)
    q, a, b = _case(workloads, n, limbs, 92000 + 10 * limbs + n)
    a[0] = 0
    b[-1] = workloads.q_minus_one(q)
    with polymul.Plan(n, 32 * limbs, limbs, q) as plan:
        primes = [int(p) for p in plan.primes()]
        beta = [int(x) for x in plan.table(polymul.TABLE_BETA, np.uint32)]
        res = plan.debug_stage(a, b, polymul.STAGE_RESIDUES).reshape(2, len(primes), n)
    av, bv = oracle.from_limbs(a), oracle.from_limbs(b)
    for k, p in enumerate(primes):
        assert [int(v) for v in res[0, k]] == [x % p for x in av], "a mod p_%d" % k
        assert [int(v) for v in res[1, k]] == [beta[k] * x % p for x in bv], "beta*b mod p_%d" % k


@pytest.mark.parametrize("n,limbs", [(16384, 3), (16384, 16), (32768, 30), (2048, 128), (16384, 129), (8192, 200),
                                     (1024, 256), (1024, 257)])
def test_products(polymul, workloads, oracle, device_memory, n, limbs):
    print("[gpu-case] short conversion products", n, limbs, flush=True)
    q, a, b = _case(workloads, n, limbs, 93000 + limbs)
    expect = oracle.kronecker_gmp(a, b, q)
    with polymul.Plan(n, 32 * limbs, limbs, q) as plan:
        assert np.array_equal(plan.multiply(a, b), expect)
        with plan.operand(b) as kept:
            assert np.array_equal(plan.multiply_operand(a, kept), expect)
        pad = np.zeros(1, dtype=np.uint32)
        pa = device_memory.upload(np.concatenate([pad, a.ravel()]))
        pb = device_memory.upload(np.concatenate([pad, b.ravel()]))
        pc = device_memory.upload(np.zeros(n * limbs + 1, dtype=np.uint32))
        try:
            plan.multiply_device(pa + 4, pb + 4, pc + 4)
            got = device_memory.download(pc, (n * limbs + 1,), np.uint32)
        finally:
            for ptr in (pa, pb, pc):
                device_memory.free(ptr)
        assert np.array_equal(got[1:].reshape(n, limbs), expect)


@pytest.mark.parametrize("n,limbs", [(4096, 1), (4096, 17), (4096, 64), (4096, 65), (4096, 128), (4096, 129),
                                     (4096, 256), (8192, 1), (8192, 32), (8192, 33), (8192, 64), (8192, 65),
                                     (8192, 128), (8192, 129), (16384, 1), (16384, 16), (16384, 17), (16384, 32),
                                     (16384, 33)])
def test_column_stages(polymul, workloads, oracle, device_memory, n, limbs):
    """Two, four and eight transform rows, where the conversion does the forward
    column stages too if a lane holds whole columns (8192 coefficients above 128
    limbs, or 64 in a batch, and 16384 above 32, or in a batch: it does not):
    alone, with one operand resident, and in a batch."""
    print("[gpu-case] conversion with column stages", n, limbs, flush=True)
    q, a, b = _case(workloads, n, limbs, 94000 + n + limbs)
    a[: n // 2] = workloads.q_minus_one(q)
    expect = oracle.kronecker_gmp(a, b, q)
    with polymul.Plan(n, 32 * limbs, limbs, q) as plan, polymul.Plan(n, 32 * limbs, limbs, q) as other:
        assert np.array_equal(plan.multiply(a, b), expect)
        with plan.operand(b) as kept:
            assert np.array_equal(plan.multiply_operand(a, kept), expect)
        pa, pb = device_memory.upload(a), device_memory.upload(b)
        pcs = [device_memory.upload(np.zeros_like(a)) for _ in range(2)]
        try:
            plan.multiply_device(pa, pb, pcs[0])
            assert np.array_equal(device_memory.download(pcs[0], a.shape, np.uint32), expect)
            polymul.multiply_device_batch([plan, other], [pa, pa], [pb, pb], pcs)
            for pc in pcs:
                assert np.array_equal(device_memory.download(pc, a.shape, np.uint32), expect)
        finally:
            for ptr in [pa, pb] + pcs:
                device_memory.free(ptr)
