"""More polynomials in one call than one launch has threads for (2^18 + 1 of 8 limbs at N = 2^13,
137 GB: a column pass of 2^32 threads and more): the first, a middle and the last polynomial
transform as alone, both ways, and those of zeros stay zero."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def hip_runtime():
    """The HIP runtime that the engine has loaded."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = C.CDLL(path)

    def call(name, *args):
        assert getattr(hip, name)(*args) == 0, name
    return call


def test_more_polynomials_than_one_launch_holds():
    import shmoai_amd as shm
    ctx = shm.Context(13, [50] * 8 + [60], 1)
    polys, limbs = (1 << 18) + 1, 8
    words = limbs * ctx.N
    hip = hip_runtime()
    free, total = C.c_size_t(), C.c_size_t()
    hip("hipMemGetInfo", C.byref(free), C.byref(total))
    if free.value < polys * words * 8 + (4 << 30):
        pytest.skip("needs 141 GB of free device memory")
    rng = np.random.default_rng(1)
    one = np.stack([rng.integers(0, int(q), size=ctx.N, dtype=np.uint64) for q in ctx.coeff_modulus[:limbs]])
    ct = shm.Ciphertext(ctx, 2, 1).load(np.concatenate([one, one]).ravel())
    ctx.ntt_forward(ct.data_ptr(), 2, limbs, 0)
    alone = ct.numpy()[:words].reshape(limbs, ctx.N)
    buf = C.c_void_p()
    hip("hipMalloc", C.byref(buf), C.c_size_t(polys * words * 8))
    try:
        at = lambda p: C.c_void_p(buf.value + p * words * 8)
        read = np.empty_like(one)

        def poly(p):
            hip("hipMemcpy", C.c_void_p(read.ctypes.data), at(p), C.c_size_t(words * 8), C.c_int(2))
            return read

        hip("hipMemset", buf, C.c_int(0), C.c_size_t(polys * words * 8))
        for p in (0, polys // 2, polys - 1):
            hip("hipMemcpy", at(p), C.c_void_p(one.ctypes.data), C.c_size_t(words * 8), C.c_int(1))
        ctx.ntt_forward(buf.value, polys, limbs, 0)
        shm.synchronize()
        for p in (0, polys // 2, polys - 1):
            assert np.array_equal(poly(p), alone), f"forward, polynomial {p}"
        assert not poly(polys - 2).any()
        ctx.ntt_inverse(buf.value, polys, limbs, 0)
        shm.synchronize()
        for p in (0, polys // 2, polys - 1):
            assert np.array_equal(poly(p), one), f"inverse, polynomial {p}"
    finally:
        hip("hipFree", buf)
