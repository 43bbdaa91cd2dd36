"""NTT of every butterfly form against the oracle, bit-exact: primes just below a power of
two take split products (the largest and smallest bit sizes they cover, and the longest
distance below the power of two that a chain of N = 2^17 holds), 60-bit and short primes
and launches that mix them the other forms; every ring degree, odd polynomial counts, and
the residues 0 and q - 1 beside random ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ring degree, primes (data, then one special prime), transformed limbs (first, count), polynomials
CASES = [
    (12, [46, 51, 36, 58, 30], 0, 4, 3),
    (13, [50, 50, 50, 60], 0, 3, 1),
    (13, [50, 60, 40, 34, 50], 0, 4, 2),
    (14, [51, 46, 46, 36, 58, 58, 51], 0, 6, 5),
    (15, [51, 46, 46, 51], 0, 3, 4),
    (16, [51, 46, 46, 50, 58, 60], 0, 4, 9),
    (16, [51, 46, 60, 50], 1, 2, 1),
    (17, [51] * 45 + [46, 60], 0, 3, 2),
    (17, [51, 46, 58, 51], 0, 3, 1),
]


@pytest.mark.parametrize("logN,bits,first,count,polys", CASES, ids=lambda v: str(len(v)) if isinstance(v, list) else str(v))
def test_ntt_forms_bitexact(oracle_lib, logN, bits, first, count, polys):
    import shmoai_amd as shm
    ctx = shm.Context(logN, bits, 1)
    ref = oracle_lib.Ref(logN, bits, 1)
    rng = np.random.default_rng(logN * 100 + len(bits))
    N = ref.N
    x = np.empty((polys, count, N), np.uint64)
    for k in range(count):
        q = int(ref.primes[first + k])
        x[:, k] = rng.integers(0, q, size=(polys, N), dtype=np.uint64)
        x[0, k, ::3] = q - 1
        x[0, k, 1::3] = 0
        x[-1, k] = np.where(rng.random(N) < 0.5, q - 1, x[-1, k])
    batch = shm.SharedABatch(ctx, max(polys - 1, 1), ctx.chain(count))  # polys x count limbs of device words
    full = np.zeros((max(polys, 2), count, N), np.uint64)
    full[:polys] = x
    batch.load(full.ravel())
    ctx.ntt_forward(batch.data_ptr(), polys, count, first)
    got = batch.numpy().reshape(full.shape)[:polys]
    exp = ref.ntt(x.ravel(), np.tile(np.arange(first, first + count), polys)).reshape(x.shape)
    assert np.array_equal(got, exp)
    ctx.ntt_inverse(batch.data_ptr(), polys, count, first)
    assert np.array_equal(batch.numpy().reshape(full.shape)[:polys], x)
    # the inverse of words that no forward transform produced
    batch.load(full.ravel())
    ctx.ntt_inverse(batch.data_ptr(), polys, count, first)
    inv = batch.numpy().reshape(full.shape)[:polys]
    back = ref.ntt(np.ascontiguousarray(inv).ravel(), np.tile(np.arange(first, first + count), polys)).reshape(x.shape)
    assert np.array_equal(back, x)
