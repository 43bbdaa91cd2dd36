"""Decoding of coefficients of every size against the oracle: those that follow from two
residues (0, small ones of both signs, up to half the product of the first two primes) and
those that need the whole composition (just above it, and near Q / 2), at one prime, at two
and at many.

Both sides run the same composition and the same FFT butterflies, in FP64: 12 stages of one
product and one sum of relative error 2^-53 each bound the difference of a slot by about
12 * 4 * 2^-53 < 1e-14 of the slots' root mean square per coefficient scale; 1e-12 of the
largest slot leaves room for the roots' own last bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ql", [1, 2, 3, 9])
@pytest.mark.parametrize("size", ["zero", "tiny", "message", "two_primes", "above_two_primes", "half_q"])
def test_decode_matches_oracle(oracle_lib, Ql, size):
    import shmoai_amd as shm
    bits = [51] + [46] * 4 + [51] * 4 + [51]
    ctx = shm.Context(13, bits, 1)
    ref = oracle_lib.Ref(13, bits, 1)
    primes = [int(q) for q in ref.primes[:Ql]]
    Q = 1
    for q in primes:
        Q *= q
    two = primes[0] * (primes[1] if Ql > 1 else 1)
    rng = np.random.default_rng(3)
    base = {"zero": [0], "tiny": [0, 1, -1, 2, -3], "message": [1 << 46, -(1 << 50), 12345, -1, 1 - (1 << 45)],
            "two_primes": [two // 2, -(two // 2), two // 2 - 1, two // 3],
            "above_two_primes": [two // 2 + 1, -(two // 2) - 1, two, -two + 5],
            "half_q": [Q // 2, -(Q // 2), Q // 2 - 7, Q // 3]}[size]
    picks = rng.integers(0, len(base), ref.N)
    limbs = np.empty((Ql, ref.N), np.uint64)
    for k, q in enumerate(primes):
        limbs[k] = np.array([b % q for b in base], np.uint64)[picks]
    pt_words = ref.ntt(limbs.ravel(), np.arange(Ql, dtype=np.uint32))
    scale = 2.0 ** 40
    pt = shm.Plaintext(ctx, ctx.chain(Ql)).load(pt_words)
    pt.scale = scale
    got = shm.Encoder(ctx).decode(pt, complex_out=True)
    re, im = ref.decode(pt_words, Ql, scale)
    want = re + 1j * im
    assert np.max(np.abs(got - want)) <= 1e-12 * max(np.max(np.abs(want)), 1e-300)


@pytest.mark.parametrize("bits", [[51] + [46] * 4 + [51], [50] * 3 + [60]], ids=["split", "mixed"])
@pytest.mark.parametrize("scale", [2.0 ** 30, 2.0 ** 58, 2.0 ** 61, 2.0 ** 90])
def test_encode_matches_oracle(oracle_lib, bits, scale):
    """Coefficients below, around and above the 2^60 up to which they travel as one signed
    word; above, each prime reduces them by itself. Whole words, bit-exact."""
    import shmoai_amd as shm
    ctx = shm.Context(13, bits, 1)
    ref = oracle_lib.Ref(13, bits, 1)
    Ql, n = len(bits) - 1, ref.N // 2
    # one slot vector with a large constant coefficient beside small ones, one with all alike
    for v in (np.concatenate([[3.75], np.zeros(n - 1)]), np.full(n, -1.625)):
        got = shm.Encoder(ctx).encode(v, scale, 1).numpy()
        assert np.array_equal(got, ref.encode(v, Ql, scale))
