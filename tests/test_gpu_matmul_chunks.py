"""Row chunks whose fragment workspaces differ: at these row counts the last chunks hold fewer
64-row steps than the first and yet take more weight fragments (their phases stage more row
blocks). One, two and four column blocks, 4 and 6 weight digits, against the 64-bit variant,
whole words; the counts beside them, whose chunks are alike, too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows, columns, prime chain, input scale, largest weight
DIGITS4 = ([50, 50, 60], 2.0 ** 30, 1.9)   # |w scale| < 127 (256^4 - 1) / 255
DIGITS6 = ([51, 46, 51], 2.0 ** 46, 0.09)  # above 127 (256^5 - 1) / 255 = 2^38.99


@pytest.mark.parametrize("chain", [DIGITS4, DIGITS6], ids=["4digits", "6digits"])
@pytest.mark.parametrize("rows,cols", [(256, 16), (257, 16), (257, 32), (384, 16), (385, 16), (385, 32), (385, 64),
                                       (386, 16), (577, 16), (578, 33), (771, 16)])
def test_row_chunks_equal_u64(chain, rows, cols):
    import shmoai_amd as shm
    bits, scale, largest = chain
    ctx = shm.Context(12, bits, 1)
    rng = np.random.default_rng(rows * 100 + cols)
    X = []
    for _ in range(rows):
        a = np.stack([rng.integers(0, int(q), size=ctx.N, dtype=np.uint64) for q in ctx.coeff_modulus[:2]] * 2)
        a[:, ::9] = (np.array([int(q) - 1 for q in ctx.coeff_modulus[:2]] * 2, np.uint64))[:, None]
        ct = shm.Ciphertext(ctx, 2, 1).load(a.ravel())
        ct.scale = scale
        X.append(ct)
    W = rng.normal(0, largest / 8, (rows, cols)).clip(-largest, largest)
    W[0, 0], W[rows - 1, cols - 1] = largest, -largest
    out = {}
    for variant in (shm.MATMUL_INT8, shm.MATMUL_U64):
        o = shm.ct_pt_matrix_mul_wo_pre(X, W, rows, cols, rows, ctx, variant=variant)
        assert shm.last_matmul_variant() == variant
        out[variant] = [c.numpy() for c in o]
    for i in range(cols):
        assert np.array_equal(out[shm.MATMUL_INT8][i], out[shm.MATMUL_U64][i]), f"output {i}"
