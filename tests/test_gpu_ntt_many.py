"""More polynomials in one call than one launch has threads for (2^18 + 1 of 8 limbs at N = 2^13,
137 GB: a column pass of 2^32 threads and more): the first, a middle and the last polynomial
transform as alone, both ways, and those of zeros stay zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_more_polynomials_than_one_launch_holds():
    import torch
    import shmoai_amd as shm
    ctx = shm.Context(13, [50] * 8 + [60], 1)
    polys, limbs = (1 << 18) + 1, 8
    if torch.cuda.mem_get_info()[0] < polys * limbs * ctx.N * 8 + (4 << 30):
        pytest.skip("needs 141 GB of free device memory")
    rng = np.random.default_rng(1)
    one = torch.from_numpy(np.stack([rng.integers(0, int(q), size=ctx.N) for q in ctx.coeff_modulus[:limbs]])).cuda()
    at = [0, polys // 2, polys - 1]
    x = torch.zeros((polys, limbs, ctx.N), dtype=torch.int64, device="cuda")
    try:
        for p in at:
            x[p] = one
        alone = one.clone()
        torch.cuda.synchronize()
        ctx.ntt_forward(alone.data_ptr(), 1, limbs, 0)
        ctx.ntt_forward(x.data_ptr(), polys, limbs, 0)
        shm.synchronize()
        for p in at:
            assert torch.equal(x[p], alone), f"forward, polynomial {p}"
        assert not x[polys - 2].any()
        ctx.ntt_inverse(x.data_ptr(), polys, limbs, 0)
        shm.synchronize()
        for p in at:
            assert torch.equal(x[p], one), f"inverse, polynomial {p}"
    finally:
        del x
        torch.cuda.empty_cache()
