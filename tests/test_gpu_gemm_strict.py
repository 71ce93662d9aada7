"""f32 / f16 weights times several vectors, tiled over rows and vectors: the
CPU path's bits (batchMatMulUnified's f32 branch, one math.matVecMul per row)
at the edges of every tile and on both sides of the choice between them."""
import numpy as np
import pytest

import mmhip as mm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = mm.Context(0)
    yield c
    c.close()


# (vectors, rows, columns); with 256 CUs: 16 x 32 tiles from 448 workgroups,
# then 8 x 16, then 4 x 16, and one workgroup per row up to 256 of them.
@pytest.mark.parametrize("n,rows,cols", [(97, 2305, 131), (32, 7168, 128), (33, 7153, 3), (49, 1001, 517), (17, 301, 1030),
                                         (64, 65, 2048), (64, 64, 2048), (16, 257, 4), (2, 300, 513)])
@pytest.mark.parametrize("t", [mm.F32, mm.F16])
def test_tiles_give_the_cpu_paths_bits(ctx, orc, t, n, rows, cols):
    rng = np.random.default_rng(n * 1000 + rows + cols)
    raw = mm.make_weight(rng, t, rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[0, 0], x[-1, -1] = np.inf, -0.0  # poisons its own vector's outputs only
    got = ctx.batch_mat_mul(raw, t, x, rows, n, cols)
    ref = orc.batch_mat_mul_unified(raw, t, x, rows, n, cols)
    np.testing.assert_array_equal(got.view(np.uint32), np.asarray(ref).reshape(n, rows).view(np.uint32))
