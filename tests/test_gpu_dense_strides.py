"""Dense operations at the edges of their kernels' tiles: contractions of
operands read at their own strides in every order (rows or k contiguous,
neither: copied first; C scattered), with the k range in parts, and aliased
with C; permutations, sums of two terms and scalar products around the 32- and
64-element tiles.  Bounds: k + 2 roundings of the sum of |a| |b| for
contractions, two roundings per term for sums, n for scalar products."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def _dev(ctx, a):
    return lt.device_array(ctx, a.shape, np.ascontiguousarray(a))


# dimension orders of A (i, a | k, c), B (k, c | j, b) and C (i, a, j, b)
ORDERS = [("iakc", "kcjb", "iajb"), ("ikac", "kjcb", "ijab"), ("kcia", "jbkc", "jbia"), ("ciak", "bkcj", "bija"),
          ("kica", "ckbj", "ajbi")]
# extents of i, a, j, b, k, c
SHAPES = [(1, 1, 1, 1, 1, 1), (3, 5, 4, 16, 2, 8), (4, 4, 8, 8, 1, 16), (5, 13, 3, 43, 3, 11), (1, 17, 1, 65, 1, 33),
          (2, 3, 2, 5, 67, 31), (11, 29, 7, 37, 5, 9), (40, 41, 32, 33, 2, 3), (1, 1, 3, 7, 9, 10)]


@pytest.mark.parametrize("zero", [True, False])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("orders", ORDERS, ids="-".join)
def test_contract2(gpu_ctx, orders, shape, zero):
    print("dense", orders, shape, zero, flush=True)
    ext = dict(zip("iajbkc", shape))
    oa, ob, oc = orders
    rng = np.random.default_rng(sum(shape))
    a, b, c = (rng.standard_normal([ext[x] for x in o]) for o in orders)
    free = [x for x in oa + ob if x not in "kc"]
    con = lt.contraction2(2, 2, 2, permc=[free.index(x) for x in oc])
    for x in "kc":
        con.contract(oa.index(x), ob.index(x))
    da, db, dc = _dev(gpu_ctx, a), _dev(gpu_ctx, b), _dev(gpu_ctx, c)
    lt.tod_contract2(con, da, db, dc, d=0.5, zero=zero)
    rule = "%s,%s->%s" % orders
    ref = 0.5 * np.einsum(rule, a, b) + (0 if zero else c)
    bound = (ext["k"] * ext["c"] + 2) * EPS * (0.5 * np.einsum(rule, abs(a), abs(b)) + abs(c))
    assert np.all(abs(dc.download() - ref) <= 2 * bound)     # both sides round


@pytest.mark.parametrize("m,n,k", [(16, 64, 5000), (33, 130, 1023), (700, 640, 257), (1300, 1300, 19)])
def test_contract2_parts_and_large(gpu_ctx, m, n, k):
    print("dense", m, n, k, flush=True)
    rng = np.random.default_rng(m)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((n, k))
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 1)
    da, db, dc = _dev(gpu_ctx, a), _dev(gpu_ctx, b), lt.device_array(gpu_ctx, (m, n))
    lt.tod_contract2(con, da, db, dc)
    assert np.all(abs(dc.download() - a @ b.T) <= 2 * (k + 2) * EPS * (abs(a) @ abs(b).T))


def test_contract2_into_operand(gpu_ctx):
    rng = np.random.default_rng(4)
    a, b = rng.standard_normal((70, 70)), rng.standard_normal((70, 70))
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 0)
    da, db = _dev(gpu_ctx, a), _dev(gpu_ctx, b)
    lt.tod_contract2(con, da, db, da)
    assert np.all(abs(da.download() - a @ b) <= 2 * 72 * EPS * (abs(a) @ abs(b)))


# C beyond 32 MiB whose contiguous dimension leads neither index well: its
# product goes through a contiguous copy, operands with short runs too
STAGED = [(("iakc", "kcjb", "bija"), (59, 5, 239, 61, 2, 3)), (("ikac", "ckbj", "ajbi"), (5, 61, 59, 239, 1, 7)),
          (("kica", "kcjb", "bija"), (59, 5, 239, 61, 2, 3)), (("kica", "kjcb", "bija"), (401, 5, 431, 5, 2, 3))]


@pytest.mark.parametrize("zero", [True, False])
@pytest.mark.parametrize("orders,shape", STAGED, ids=str)
def test_contract2_into_short_runs(gpu_ctx, orders, shape, zero):
    test_contract2(gpu_ctx, orders, shape, zero)


# (from 2^20 elements on tiles are 64 wide where the shorter side has 33 to 63
# elements, and in scalar products where both are beyond 32; from 2^22 on they
# are stored past the caches, short rows that adjoin as one run)
@pytest.mark.parametrize("dims", [(31, 3, 33), (32, 32), (33, 2, 33), (63, 65), (64, 3, 64), (130, 2, 67), (1, 200), (9, 1, 7, 40),
                                  (65, 63, 65), (33, 300, 33), (64, 65, 64), (130, 40, 67), (163, 161, 163), (1100, 31, 130),
                                  (33, 970, 33), (63, 270, 63), (40, 660, 41), (41, 2600, 41), (9, 52000, 9)], ids=str)
def test_permutes_sums_products(gpu_ctx, dims):
    print("permute", dims, flush=True)
    rng = np.random.default_rng(len(dims))
    n = len(dims)
    perm = list(range(n))[::-1]
    x = rng.standard_normal(dims)
    dx = _dev(gpu_ctx, x)
    xt = x.transpose(perm)
    out = lt.device_array(gpu_ctx, xt.shape)
    lt.tod_copy(dx, out, perm, -0.5)
    assert np.array_equal(out.download(), -0.5 * xt)
    lt.tod_copy(dx, out, perm, 0.25, zero=False)
    assert np.all(abs(out.download() + 0.25 * xt) <= EPS * abs(xt))
    if dims == dims[::-1]:
        y = rng.standard_normal(dims)
        dy = _dev(gpu_ctx, y)
        for p, q in [(None, perm), (perm, None), (perm, perm)]:
            lt.tod_add([(dx, p, 0.75), (dy, q, -0.3)], out)
            u, v = 0.75 * (x if p is None else xt), -0.3 * (y if q is None else y.transpose(perm))
            assert np.all(abs(out.download() - (u + v)) <= 2 * EPS * (abs(u) + abs(v)))
    y = rng.standard_normal(xt.shape)
    r = lt.tod_dotprod(dx, _dev(gpu_ctx, y), perm, None)
    assert abs(r - np.vdot(xt, y)) <= 2 * x.size * EPS * np.vdot(abs(xt), abs(y))


@pytest.mark.parametrize("dims,perm", [((70, 61, 1009), (1, 0, 2)), ((50000, 9, 11), (0, 2, 1)), ((3000, 33, 45), (0, 2, 1))], ids=str)
def test_past_the_caches(gpu_ctx, dims, perm):
    x = np.random.default_rng(5).standard_normal(dims)
    ref = x.transpose(perm)
    dx, out = _dev(gpu_ctx, x), lt.device_array(gpu_ctx, ref.shape)
    lt.tod_copy(dx, out, perm, 3.0)
    assert np.array_equal(out.download(), 3.0 * ref)
    lt.tod_copy(dx, out, perm, -1.0, zero=False)
    # 3 x is rounded, and 3 x - x: at most (3 + 2) u |x|
    assert np.all(abs(out.download() - 2.0 * ref) <= 5 * EPS * abs(ref) * (1 + EPS))
