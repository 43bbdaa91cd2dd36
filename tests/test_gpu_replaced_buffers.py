"""Calls that give a ciphertext or batch a new block (Chebyshev evaluation, level raising,
shared-a rotation) on a created stream return the old one behind that stream's work: a block
that came from the default stream, with kernels of the call still reading it, is not the next
one that the default stream hands out. A spare block of the same size waits on the default
stream's list, so that the next object there takes the spare one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BITS = [51] + [46] * 3 + [51] * 8 + [51] * 4
SCALE = 2.0 ** 46


@pytest.fixture(scope="module")
def env():
    import shmoai_amd as shm
    ctx = shm.Context(13, BITS, 4)
    sk = shm.SecretKey(ctx, seed=5, hamming_weight=64)
    keys = shm.SharedAKeys(ctx, sk, 3, 64, 77, ctx.chain(4))
    keys.add_galois([3], seed=9)
    return shm, ctx, sk, keys, sk.gen_relinkey(seed=3)


def words(ctx, polys, Ql, seed):
    rng = np.random.default_rng(seed)
    return np.stack([rng.integers(0, int(q), size=ctx.N, dtype=np.uint64)
                     for q in ctx.coeff_modulus[:Ql]] * polys).ravel()


@pytest.mark.parametrize("op", ["chebyshev", "batch_modraise", "batch_rotate"])
def test_old_block_is_returned_on_the_calls_stream(env, op):
    shm, ctx, sk, keys, rk = env
    ev = shm.Evaluator(ctx)
    if op == "chebyshev":
        Ql, polys = 12, 2
        make = lambda: shm.Ciphertext(ctx, 2, ctx.chain(Ql))
        call = lambda x, st: ev.evaluate_chebyshev_inplace([x], [0.5, 0.25, 0.125], -1.0, 1.0, rk, stream=st)
    elif op == "batch_modraise":
        Ql, polys = 1, 4
        make = lambda: shm.SharedABatch(ctx, 3, ctx.chain(1))
        call = lambda x, st: x.modraise_inplace(stream=st)
    else:
        Ql, polys = 4, 4
        make = lambda: shm.SharedABatch(ctx, 3, ctx.chain(4))
        call = lambda x, st: keys.rotate_inplace(x, 3, stream=st)
    a = words(ctx, polys, Ql, 1)

    def loaded():
        x = make().load(a)
        x.scale = SCALE
        return x

    want = loaded()
    call(want, None)  # on the default stream; builds tables
    expect = want.numpy()
    st = shm.Stream()
    x = loaded()
    old = x.data_ptr()
    spare = make()
    del spare
    call(x, st.h)
    fresh = make()
    assert fresh.data_ptr() != old
    fresh.load(words(ctx, polys, Ql, 2))
    shm.synchronize(st.h)
    assert np.array_equal(x.numpy(), expect)
    del x, fresh
    st.close()
