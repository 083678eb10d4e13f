"""The split-precision product's workgroup tiles (48 x 64) at the edges of
their row and column panels and 64-k chunks, one or several pairs per C block,
for every slice count: exact on small integers, and against the wave tiles'
sums of the same slice products (2 (S + 1) roundings of the sum of |a| |b| on
either side) on random matrices."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu


def _tensor(ctx, dims, splits):
    bis = lt.block_index_space(dims)
    for d, points in enumerate(splits):
        for p in points:
            bis.split([1 if i == d else 0 for i in range(len(dims))], p)
    return lt.block_tensor(ctx, bis)


def _run(ctx, a, b, splits, slices, tile):
    sm, sn, sk = splits
    bta, btb = _tensor(ctx, a.shape, (sm, sk)), _tensor(ctx, b.shape, (sk, sn))
    bta.from_dense(a)
    btb.from_dense(b)
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 0)
    op = lt.btod_contract2(con, bta, btb)
    op.set_ozaki(slices)
    op.set_ozaki_tile(tile)
    c = _tensor(ctx, (a.shape[0], b.shape[1]), (sm, sn))
    op.perform(c, lt.LT_MODE_OZAKI)
    return c.to_dense()


SHAPES = [((1, 1, 1), ((), (), ())), ((16, 64, 64), ((), (), ())), ((17, 65, 65), ((), (), ())),
          ((33, 63, 130), ((), (), ())), ((48, 129, 200), ((), (), (64,))), ((97, 70, 150), ((49,), (5,), (1, 66))),
          ((113, 191, 63), ((48, 100), (64,), (31, 32)))]


@pytest.mark.parametrize("slices", range(1, 9))
@pytest.mark.parametrize("shape,splits", SHAPES, ids=[str(s[0]) for s in SHAPES])
def test_workgroup_tiles(gpu_ctx, shape, splits, slices):
    m, n, k = shape
    print("split", shape, splits, slices, flush=True)
    rng = np.random.default_rng(m + n + k)
    a, b = rng.integers(-60, 61, (m, k)).astype(float), rng.integers(-60, 61, (k, n)).astype(float)
    assert np.array_equal(_run(gpu_ctx, a, b, splits, slices, 2), a @ b)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    d = _run(gpu_ctx, a, b, splits, slices, 2) - _run(gpu_ctx, a, b, splits, slices, 0)
    assert np.all(abs(d) <= 4 * (slices + 1) * 2.0 ** -53 * (abs(a) @ abs(b)))
