"""ModDown merged with the rescale (relinearised products inside polynomial evaluation), whole
words against exact centred divisions in Python integers: 2 to 5 special primes, so conversions
of 3 to 6 source limbs, at ring degrees whose column stages take one round and two, the last
digit shorter than the others.

The product is reached through the Chebyshev series c_2 T_2(x) on [-1, 1]: the affine map is
one times x (its rescale drops a limb exactly), T_2 = 2 x x - 1 is the product under test, and
the sum of one term is a constant product and a rounded rescale."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ring degree, special primes, data primes
CASES = [(12, 2, 6), (13, 3, 9), (12, 4, 8), (13, 4, 8), (12, 5, 10), (13, 5, 10), (14, 5, 10),
         (16, 5, 15)]  # 18 limbs: the raised digits' row stages fused with the key products


def centred(limbs, primes):
    """The integer of least magnitude with these residues, per coefficient."""
    D = 1
    for q in primes:
        D *= q
    x = sum(v.astype(object) * (D // q * pow(D // q, -1, q)) for v, q in zip(limbs, primes)) % D
    return np.where(x > D // 2, x - D, x)


@pytest.mark.parametrize("logN,nP,nQ", CASES)
def test_merged_moddown_rescale_exact(oracle_lib, logN, nP, nQ):
    import shmoai_amd as shm
    bits = [51] + [46] * (nQ - 1) + [51] * nP
    ctx, ref = shm.Context(logN, bits, nP), oracle_lib.Ref(logN, bits, nP)
    sk = shm.SecretKey(ctx, seed=5, hamming_weight=64)
    rk = ref.gen_relin_key(ref.sk_ntt(ref.sample_ternary(5, 64)), 8).reshape(-1, 2, nQ + nP, ref.N)
    primes = [int(q) for q in ref.primes]
    N, top, scale, c2 = ref.N, nQ - 1, 2.0 ** 46, 0.7310585786
    rng = np.random.default_rng(logN + nP)
    x = np.stack([rng.integers(0, q, size=N, dtype=np.uint64) for q in primes[:top]] * 2)
    for k in range(2 * top):  # the largest residue among the random ones
        x[k, ::5] = primes[k % top] - 1
    ct = shm.Ciphertext(ctx, 2, ctx.chain(top)).load(x.ravel())
    ct.scale = scale
    shm.Evaluator(ctx).evaluate_chebyshev_inplace(ct, [0.0, 0.0, c2], -1.0, 1.0, sk.gen_relinkey(seed=8))

    L = top - 1                                       # limbs of the product's operands
    xs = x.reshape(2, top, N)[:, :L]
    d = ref.tensor(np.ascontiguousarray(xs).ravel(), np.ascontiguousarray(xs).ravel(), L).reshape(3, L, N)
    ext = list(range(L)) + list(range(nQ, nQ + nP))   # primes of the raised polynomials
    q_of = [primes[p] for p in ext]
    d = [[2 * d[i][k].astype(object) % primes[k] for k in range(L)] for i in range(3)]
    as_words = lambda rows: np.stack([np.array(r, np.uint64) for r in rows])
    to_ntt = lambda v, idx: ref.ntt(as_words([v % primes[p] for p in idx]).ravel(), np.array(idx, np.uint32)).reshape(-1, N)
    coef = lambda rows, idx: ref.intt(as_words(rows).ravel(), np.array(idx, np.uint32)).reshape(-1, N)
    c2coef = coef(d[2], range(L))
    P = 1
    for p in primes[nQ:]:
        P *= p
    acc = [[P * d[o][k] % primes[k] if k < L else 0 for k in range(L + nP)] for o in range(2)]
    for g in range(-(-L // nP)):
        own = list(range(g * nP, min((g + 1) * nP, L)))
        raised = to_ntt(centred(c2coef[own], [primes[k] for k in own]), ext)
        for o in range(2):
            for k, p in enumerate(ext):
                acc[o][k] = (acc[o][k] + raised[k].astype(object) * rk[g, o, p].astype(object)) % q_of[k]
    B = P * primes[L - 1]
    t2, last = [], list(range(L - 1, L + nP))         # the limbs divided away
    for o in range(2):
        delta = to_ntt(centred(coef([acc[o][k] for k in last], [ext[k] for k in last]), [q_of[k] for k in last]),
                       range(L - 1))
        t2.append([(acc[o][k] - delta[k].astype(object)) * pow(B, -1, primes[k]) % primes[k] for k in range(L - 1)])
    L -= 1
    s2 = scale * scale / float(primes[L])
    minus_one = -round(s2)
    K = round(c2 * (scale * float(primes[L - 1]) / s2))
    want = []
    for o in range(2):
        v = [K * (t2[o][k] + (minus_one if o == 0 else 0)) % primes[k] for k in range(L)]
        delta = to_ntt(centred(coef(v[L - 1:], [L - 1]), [primes[L - 1]]), range(L - 1))
        want.append(as_words([(v[k] - delta[k].astype(object)) * pow(primes[L - 1], -1, primes[k]) % primes[k]
                              for k in range(L - 1)]))
    assert ct.coeff_modulus_size == L - 1
    assert np.array_equal(ct.numpy(), np.stack(want).ravel())
