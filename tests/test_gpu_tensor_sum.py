"""Sums of ciphertext products, 15 per launch (the column packing's inner sums), bit-exact
against the oracle: one launch, a full one, one product and a full launch beyond it, on a
chain of 46- to 51-bit primes (split sums) and on one with a 60-bit prime (single products)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [1, 2, 15, 16, 31])
@pytest.mark.parametrize("bits", [[51, 46, 46, 51], [60, 40, 40, 60]], ids=["split", "single"])
def test_tensor_sum_bitexact(oracle_lib, bits, cols):
    import shmoai_amd as shm
    ctx = shm.Context(12, bits, 1)
    ref = oracle_lib.Ref(12, bits, 1)
    rng = np.random.default_rng(cols)
    sk = shm.SecretKey(ctx, seed=1, hamming_weight=64)
    s_ref = ref.sk_ntt(ref.sample_ternary(1, 64))
    Ql = 3

    def words():
        a = np.stack([rng.integers(0, int(q), size=ref.N, dtype=np.uint64) for q in ref.primes[:Ql]] * 2)
        for k in range(2 * Ql):  # the largest residue among the random ones
            a[k, ::3] = int(ref.primes[k % Ql]) - 1
        return a.ravel()

    xs, ws = [words() for _ in range(cols)], [words() for _ in range(cols)]
    X, W = ([shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(v) for v in vs] for vs in (xs, ws))
    for ct in X + W:
        ct.scale = 2.0 ** 40
    out = shm.ct_ct_matrix_mul_colpacking(X, W, sk.create_galois_keys_from_steps([1], seed=9), sk.gen_relinkey(seed=5),
                                          ctx, cols, 1, cols, 1, 0)
    exp = ref.ctct_matmul_colpacking(xs, ws, Ql, 1, 0, {}, ref.gen_relin_key(s_ref, 5))
    assert np.array_equal(out[0].numpy(), exp[0])


@pytest.mark.parametrize("square", [False, True])
def test_product_written_in_place_bitexact(oracle_lib, square):
    """The first product replaces the two-polynomial buffer, the second (after relinearisation)
    is written into the room for three."""
    import shmoai_amd as shm
    bits = [51, 46, 46, 51]
    ctx = shm.Context(12, bits, 1)
    ref = oracle_lib.Ref(12, bits, 1)
    rng = np.random.default_rng(3)
    sk = shm.SecretKey(ctx, seed=1, hamming_weight=64)
    s_ref = ref.sk_ntt(ref.sample_ternary(1, 64))
    rk, rkey = sk.gen_relinkey(seed=5), ref.gen_relin_key(s_ref, 5)
    a, b = (np.stack([rng.integers(0, int(q), size=ref.N, dtype=np.uint64) for q in ref.primes[:3]] * 2).ravel()
            for _ in range(2))
    ev = shm.Evaluator(ctx)
    ct, other = shm.Ciphertext(ctx, 2, ctx.chain(3)).load(a), shm.Ciphertext(ctx, 2, ctx.chain(3)).load(b)
    for _ in range(2):
        ev.multiply_inplace(ct, ct if square else other)
        a = ref.tensor(a, a if square else b, 3)
        assert np.array_equal(ct.numpy(), a)
        ev.relinearize_inplace(ct, rk)
        a = ref.relinearize(a, 3, rkey)
        assert np.array_equal(ct.numpy(), a)
