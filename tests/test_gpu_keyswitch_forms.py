"""Key switching over the forms of the base conversions, bit-exact against the oracle: 1 to 5
source limbs fused into the NTT's column stages at every ring degree (column stages of one
and of two rounds), a last digit shorter than the others, and chains outside the fused form
(60-bit primes, more than 5 special primes). Conversions of 6 source limbs come from ModDown
merged with the rescale (test_gpu_merged_rescale.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ring degree, prime sizes, special primes, level
CASES = [
    (12, [51] + [46] * 3 + [51] * 2 + [51, 51], 2, 5),
    (13, [51] + [46] * 3 + [51] * 5 + [51] * 3, 3, 7),
    (13, [50] * 4 + [60], 1, 4),
    (14, [46] * 8 + [51] * 4, 4, 6),
    (14, [50] * 4 + [60] * 2, 2, 3),
    (15, [51] + [46] * 9 + [51] * 5, 5, 7),
    (13, [46] * 12 + [51] * 6, 6, 8),
    (16, [51] + [46] * 9 + [51] * 5, 5, 10),
    (17, [51] + [46] * 3 + [51] * 2, 2, 3),
    (16, [40] * 3 + [50], 1, 3),
    # 16 rows of limbs and more: row stages fused with the products (7 digits; a last digit of one)
    (16, [51] + [46] * 13 + [51, 51], 2, 14),
    (16, [51] + [46] * 15 + [51] * 4, 4, 13),
    # as many digits as the split sums of the fused products hold
    (16, [51] * 17, 1, 16),
]


@pytest.mark.parametrize("logN,bits,nP,Ql", CASES, ids=lambda v: str(len(v)) if isinstance(v, list) else str(v))
def test_keyswitch_forms_bitexact(oracle_lib, logN, bits, nP, Ql):
    import shmoai_amd as shm
    ctx = shm.Context(logN, bits, nP)
    ref = oracle_lib.Ref(logN, bits, nP)
    rng = np.random.default_rng(logN * 10 + nP)
    sk = shm.SecretKey(ctx, seed=5, hamming_weight=64)
    gk, rk = sk.create_galois_keys_from_steps([1], seed=7), sk.gen_relinkey(seed=8)
    s_ref = ref.sk_ntt(ref.sample_ternary(5, 64))
    elt = ref.elt(1)
    gkey = ref.gen_galois_key(s_ref, elt, ref.splitmix64(7, elt))
    rkey = ref.gen_relin_key(s_ref, 8)

    def words():
        return np.stack([rng.integers(0, int(q), size=ref.N, dtype=np.uint64) for q in ref.primes[:Ql]] * 2)

    a, b = words(), words()
    for k in range(Ql):  # the largest residue among the random ones
        a[k, ::5] = a[Ql + k, ::7] = int(ref.primes[k]) - 1
    a, b = a.ravel(), b.ravel()
    ev = shm.Evaluator(ctx)
    ct = shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(a)
    ev.rotate_vector_inplace(ct, 1, gk)
    assert np.array_equal(ct.numpy(), ref.rotate(a, Ql, elt, gkey))
    ct = shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(a)
    ev.multiply_inplace(ct, shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(b))
    ev.relinearize_inplace(ct, rk)
    exp = ref.relinearize(ref.tensor(a, b, Ql), Ql, rkey)
    assert np.array_equal(ct.numpy(), exp)
    ev.rescale_to_next_inplace(ct)
    assert np.array_equal(ct.numpy(), ref.rescale(exp, Ql))
