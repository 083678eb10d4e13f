"""Permute launches over blocks of mixed sizes: lists of gathers only, and lists
whose transposing items are 32 wide, 64 wide, or some of each, with their
remainders, written and added."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

# extents, split points: blocks whose tiles are 32 or 64 wide (shorter side 33 to
# 63, blocks from 2^18 elements on in lists from 2^20 on)
CASES = [((31, 12, 33), ([7], [], [16])),
         ((72, 74, 70), ([5], [9], [])),
         ((66, 65, 64), ([], [], [])),
         ((131, 33, 97), ([33], [1], [64])),
         ((45, 560, 42), ([], [20], [])),
         # from 2^22 elements on: stores past the caches, short rows as runs
         ((170, 160, 165), ([40], [], [100])), ((5000, 90, 11), ([100], [40], [])), ((62, 1100, 63), ([], [30], []))]
PERMS = [(2, 1, 0), (1, 2, 0), (0, 2, 1), (1, 0, 2)]


def _tensor(ctx, dims, splits, data=None):
    bis = lt.block_index_space(dims)
    for i, points in enumerate(splits):
        for p in points:
            bis.split([1 if j == i else 0 for j in range(3)], p)
    t = lt.block_tensor(ctx, bis)
    if data is not None:
        t.from_dense(data)
    return t


@pytest.mark.parametrize("perm", PERMS, ids=str)
@pytest.mark.parametrize("dims,splits", CASES, ids=lambda x: str(x))
def test_copy_and_add(gpu_ctx, dims, splits, perm):
    print("permute lists", dims, splits, perm, flush=True)
    rng = np.random.default_rng(sum(dims))
    x, y = rng.standard_normal(dims), rng.standard_normal([dims[p] for p in perm])
    sp = [splits[p] for p in perm]
    a, b = _tensor(gpu_ctx, dims, splits, x), _tensor(gpu_ctx, y.shape, sp, y)
    r = _tensor(gpu_ctx, y.shape, sp)
    xt = x.transpose(perm)
    lt.btod_copy(a, r, perm, -0.5)
    assert np.array_equal(r.to_dense(), -0.5 * xt)
    lt.btod_copy(a, r, perm, 2.0, add=True, d=0.5)
    assert np.all(abs(r.to_dense() - 0.5 * xt) <= 2.0 ** -53 * abs(xt))
    lt.btod_add([(a, perm, 0.75), (b, None, -0.3)], r)
    u, v = 0.75 * xt, -0.3 * y
    # one rounding of each term and of the sum, on both sides
    assert np.all(abs(r.to_dense() - (u + v)) <= 4 * 2.0 ** -53 * (abs(u) + abs(v)))
    assert abs(lt.btod_dotprod(a, b, perm, None) - np.vdot(xt, y)) <= 2 * x.size * 2.0 ** -53 * np.vdot(abs(xt), abs(y))
