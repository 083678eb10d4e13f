"""Scalar products of operands in different orders on both sides of the rule
that reads a transposed operand by tiles or element by element: short and long
rows at either end, swapped neighbours, around the sizes where the rule turns."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

CASES = [((n, 2 ** 19 // n ** 2 + 9, n), (2, 1, 0)) for n in (7, 8, 11, 12, 31, 33)]
CASES += [((n, 80000), (1, 0)) for n in (7, 8, 24, 25)] + [((80000, n), (1, 0)) for n in (7, 8, 24, 25)]
CASES += [((2 ** 19 // n ** 2 + 1, n, n), (0, 2, 1)) for n in (44, 45, 46, 65)]
CASES += [((725, 724), (1, 0)), ((724, 724), (1, 0)), ((725, 5, 145), (2, 0, 1)), ((3, 5, 2, 7, 4), (4, 2, 0, 3, 1)),
          ((2100, 2000), (0, 1)), ((4100, 1025), (0, 1)), ((129, 257, 129), (1, 0, 2)),
          ((25, 6800, 25), (2, 1, 0)), ((22, 8700, 22), (2, 1, 0)), ((2050, 2050), (1, 0)), ((33, 3860, 33), (2, 1, 0))]


@pytest.mark.parametrize("dims,perm", CASES, ids=str)
def test_product(gpu_ctx, dims, perm):
    print("scalar product", dims, perm, flush=True)
    rng = np.random.default_rng(sum(dims))
    inv = np.argsort(perm)
    x = rng.standard_normal(dims)
    y = rng.standard_normal([dims[p] for p in perm])
    dx, dy = (lt.device_array(gpu_ctx, v.shape, v) for v in (x, y))
    for r, u in ((lt.tod_dotprod(dx, dy, perm, None, 0.5), 0.5), (lt.tod_dotprod(dy, dx, list(inv), None, -2.0), -2.0),
                 (lt.tod_dotprod(dx, dy, None, list(inv)), 1.0)):
        xt = x.transpose(perm)
        assert abs(r - u * np.vdot(xt, y)) <= 2 * x.size * 2.0 ** -53 * abs(u) * np.vdot(abs(xt), abs(y))


@pytest.mark.parametrize("n", [7, 12, 33, 70])
def test_blocks(gpu_ctx, n):
    """Blocks above and below the line in one product."""
    dims, points = (n, 2 ** 19 // n ** 2 + 40, n + 2), ([], [30], [2])
    perm = (2, 1, 0)

    def tensor(d, p, data):
        bis = lt.block_index_space(d)
        for i in range(3):
            for x in p[i]:
                bis.split([int(j == i) for j in range(3)], x)
        t = lt.block_tensor(gpu_ctx, bis)
        t.from_dense(data)
        return t
    rng = np.random.default_rng(n)
    x, y = rng.standard_normal(dims), rng.standard_normal([dims[p] for p in perm])
    a, b = tensor(dims, points, x), tensor(y.shape, [points[p] for p in perm], y)
    xt = x.transpose(perm)
    for i in range(2):
        assert abs(lt.btod_dotprod(a, b, perm, None) - np.vdot(xt, y)) <= 2 * x.size * 2.0 ** -53 * np.vdot(abs(xt), abs(y))
