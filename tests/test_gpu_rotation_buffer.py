"""Rotations stay in the caller's buffer: the public in-place calls keep the ciphertext's
address and room, so that a view of its words stays valid, nothing is returned to the block
pool while kernels read it, and a recorded rotation neither allocates its result nor frees
its input. At N = 2^16 with 16 limbs (data and special) the row stages run fused with the key
products, with 5 they run apart; every result is bit-exact against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BITS = [51] + [46] * 9 + [51] * 5 + [51] * 5


@pytest.fixture(scope="module")
def env(oracle_lib):
    import shmoai_amd as shm
    ctx, ref = shm.Context(16, BITS, 5), oracle_lib.Ref(16, BITS, 5)
    sk = shm.SecretKey(ctx, seed=5, hamming_weight=192)
    gk = sk.create_galois_keys_from_steps([1, 0], seed=7)
    s_ref = ref.sk_ntt(ref.sample_ternary(5, 192))
    keys = {e: ref.gen_galois_key(s_ref, e, ref.splitmix64(7, e)) for e in (ref.elt(1), ref.elt(0))}
    return shm, ctx, ref, gk, keys


def words(ref, Ql, seed):
    rng = np.random.default_rng(seed)
    a = np.stack([rng.integers(0, int(q), size=ref.N, dtype=np.uint64) for q in ref.primes[:Ql]] * 2)
    for k in range(2 * Ql):  # the largest residue among the random ones
        a[k, ::7] = int(ref.primes[k % Ql]) - 1
    return a.ravel()


def ops(shm, ctx, ref, gk):
    ev = shm.Evaluator(ctx)
    return {"rotate": (ref.elt(1), lambda ct, st: ev.rotate_vector_inplace(ct, 1, gk, stream=st)),
            "galois": (ref.elt(1), lambda ct, st: ev.apply_galois_inplace(ct, ref.elt(1), gk, stream=st)),
            "conjugate": (ref.elt(0), lambda ct, st: ev.complex_conjugate_inplace(ct, gk, stream=st))}


@pytest.mark.parametrize("Ql", [11, 3])
@pytest.mark.parametrize("op", ["rotate", "galois", "conjugate"])
def test_rotation_on_a_created_stream_keeps_the_buffer(env, op, Ql):
    """A ciphertext made on the default stream and rotated on a created one, with default-stream
    ciphertexts of the same size made and filled while the rotation runs."""
    shm, ctx, ref, gk, keys = env
    elt, call = ops(shm, ctx, ref, gk)[op]
    a, other = words(ref, Ql, 1), words(ref, Ql, 2)
    warm = shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(other)
    call(warm, None)  # builds the permutation table
    st = shm.Stream()
    ct = shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(a)
    at = ct.data_ptr()
    call(ct, st.h)
    spare = [shm.Ciphertext(ctx, 2, ctx.chain(Ql)) for _ in range(3)]
    for s in spare:
        assert s.data_ptr() != at
        s.load(other)
    shm.synchronize(st.h)
    assert ct.data_ptr() == at
    assert np.array_equal(ct.numpy(), ref.rotate(a, Ql, elt, keys[elt]))
    del ct, spare
    st.close()


def test_room_for_a_product_stays(env):
    """A buffer with room for three polynomials keeps it: the product after a rotation is
    written at the same address."""
    shm, ctx, ref, gk, keys = env
    Ql, ev = 11, shm.Evaluator(ctx)
    a, b = words(ref, Ql, 3), words(ref, Ql, 4)
    ct = shm.Ciphertext(ctx, 3, ctx.chain(Ql))
    at = ct.data_ptr()
    src = shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(a)
    shm.check(shm.capi.load().shm_ciphertext_copy(src.h, ct.h, None))
    ev.rotate_vector_inplace(ct, 1, gk)
    ev.multiply_inplace(ct, shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(b))
    assert ct.data_ptr() == at
    elt = ref.elt(1)
    assert np.array_equal(ct.numpy(), ref.tensor(ref.rotate(a, Ql, elt, keys[elt]), b, Ql))


def test_recorded_rotation_replays(env):
    """Recorded after one eager run on its stream, replayed three times with other work and a
    cleared output in between; the buffer is the same before, inside and after."""
    shm, ctx, ref, gk, keys = env
    Ql, ev, L = 11, shm.Evaluator(ctx), shm.capi.load()
    elt = ref.elt(1)
    a = words(ref, Ql, 5)
    X, W = shm.Ciphertext(ctx, 2, ctx.chain(Ql)).load(a), shm.Ciphertext(ctx, 2, ctx.chain(Ql))
    at = W.data_ptr()
    st = shm.Stream()

    def sequence():
        shm.check(L.shm_ciphertext_copy(X.h, W.h, st.h))
        ev.rotate_vector_inplace(W, 1, gk, stream=st.h)

    sequence()
    shm.synchronize(st.h)
    expect = ref.rotate(a, Ql, elt, keys[elt])
    assert np.array_equal(W.numpy(), expect)
    g = shm.Graph(st)
    g.begin()
    sequence()
    g.end()
    assert W.data_ptr() == at
    spare = X.copy()
    for rep in range(3):
        W.load(np.zeros_like(expect))
        g.launch()
        ev.rotate_vector_inplace(spare, 1, gk)  # unrelated default-stream work
        shm.synchronize(st.h)
        shm.synchronize(None)
        assert np.array_equal(W.numpy(), expect), f"replay {rep}"
    g.close()
    st.close()
