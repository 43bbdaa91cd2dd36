"""Rotations of several ciphertexts by one step (the column packing's), fused with their key
products: every member reads its own limbs and its added part through the permutation. From
2048 rows of 512 words over members and limbs on (4 members of 4 limbs at N = 2^16); one and
two special primes, a full batch's remainder, bit-exact against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,nP,Ql,cols", [([51, 46, 46, 51], 1, 3, 4), ([51, 46, 46, 51], 1, 3, 35),
                                             ([51] + [46] * 3 + [51] * 2, 2, 3, 5)])
def test_rotate_many_fused_bitexact(oracle_lib, bits, nP, Ql, cols):
    import shmoai_amd as shm
    ctx, ref = shm.Context(16, bits, nP), oracle_lib.Ref(16, bits, nP)
    sk = shm.SecretKey(ctx, seed=1, hamming_weight=192)
    s_ref = ref.sk_ntt(ref.sample_ternary(1, 192))
    rng = np.random.default_rng(cols)

    def words():
        a = np.stack([rng.integers(0, int(q), size=ref.N, dtype=np.uint64) for q in ref.primes[:Ql]] * 2)
        for k in range(2 * Ql):  # the largest residue among the random ones
            a[k, ::3] = int(ref.primes[k % Ql]) - 1
        return a.ravel()

    xs, ws = [words() for _ in range(cols)], [words() for _ in range(cols)]
    X, W = ([shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(v) for v in vs] for vs in (xs, ws))
    for ct in X + W:
        ct.scale = 2.0 ** 40
    gkey = {7: ref.gen_galois_key(s_ref, ref.elt(7), ref.splitmix64(9, ref.elt(7)))}
    out = shm.ct_ct_matrix_mul_colpacking(X, W, sk.create_galois_keys_from_steps([7], seed=9), sk.gen_relinkey(seed=5),
                                          ctx, cols, 2, cols, 2, 7)
    exp = ref.ctct_matmul_colpacking(xs, ws, Ql, 2, 7, gkey, ref.gen_relin_key(s_ref, 5))
    for i in range(2):
        assert np.array_equal(out[i].numpy(), exp[i]), f"output {i}"
    for w, v in zip(W, ws):  # the inputs are left as they were
        assert np.array_equal(w.numpy(), v)
