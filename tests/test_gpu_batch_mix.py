"""Batches whose products differ: every product has its own N, limbs, modulus
and operands, so that blocks of one launch run different variants side by side
and an entry that read another's parameters would show, and every output starts
as a sentinel, so that one that is never written shows.  From one product, whose
conversion is spread over the GPU, to many, which share it; the variants of the
conversion (one to eight K steps, one, two and four rows), packing and the
conversion GEMM, all row counts' transforms, both reconstructions by lanes and
the one by waves.  Bit-exact against the oracle, so there is no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIXES = {
    "one wide": [(4096, 128)],
    "one tiny": [(64, 128)],
    "one of two rows and few limbs": [(4096, 3)],
    "two alike": [(2048, 100), (2048, 100)],
    "short and long": [(64, 5), (1024, 300), (8192, 16)],
    "rows": [(2048, 9), (4096, 17), (8192, 33), (16384, 8), (32768, 4), (4096, 66), (8192, 65)],
    "edges of the variants": [(128, 16), (256, 17), (512, 32), (1024, 33), (2048, 64), (4096, 65), (4096, 128),
                              (2048, 129), (1024, 60), (1024, 61), (512, 124), (512, 125), (512, 252), (256, 253)],
    "many": [(1 << (5 + k % 8), 1 + (37 * k) % 131) for k in range(40)],
}
SENTINEL = 0xDEADBEEF


@pytest.mark.parametrize("name", list(MIXES))
def test_mixed_batch(polymul, workloads, oracle, device_memory, name):
    print("[gpu-case] mixed batch", name, flush=True)
    rng = np.random.default_rng(99000 + len(name))
    plans, ptrs, shapes, expect = [], [], [], []
    try:
        for n, limbs in MIXES[name]:
            q = workloads.random_modulus(limbs, rng)
            a, b = workloads.uniform_below(q, n, rng), workloads.uniform_below(q, n, rng)
            a[0] = workloads.q_minus_one(q)
            plans.append(polymul.Plan(n, 32 * limbs, limbs, q))
            ptrs.append([device_memory.upload(x) for x in (a, b, np.full_like(a, SENTINEL))])
            shapes.append(a.shape)
            expect.append(oracle.kronecker_gmp(a, b, q))
        for order in (1, -1):  # forwards, and backwards into fresh sentinels
            for p, shape in zip(ptrs, shapes):
                device_memory.write(p[2], np.full(shape, SENTINEL, dtype=np.uint32))
            polymul.multiply_device_batch(plans[::order], *[[p[i] for p in ptrs][::order] for i in range(3)])
            for k, (p, shape) in enumerate(zip(ptrs, shapes)):
                assert np.array_equal(device_memory.download(p[2], shape, np.uint32), expect[k]), (k, MIXES[name][k])
    finally:
        for plan in plans:
            plan.close()
        for p in ptrs:
            for ptr in p:
                device_memory.free(ptr)
