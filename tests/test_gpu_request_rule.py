"""Requests whose plans are made without timing, merged into one launch: the
kernel on both sides of the FLOP line between 32 x 64 and 64 x 64 tiles, plain
and accumulated, and fixed configurations of every kind (workgroup tiles, and
stacked kernels that merged launches run by their split-K form)."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def _operation(ctx, m, n, k, seed, tile=None):
    """Matrices with rows and k in uneven blocks, k beyond the length at which tiles are cut."""
    rng = np.random.default_rng(seed)
    out = []
    for shape, splits in (((m, k), ([m // 3], [k // 4, k // 2])), ((k, n), ([k // 4, k // 2], [])), ((m, n), ([m // 3], []))):
        bis = lt.block_index_space(shape)
        for i, points in enumerate(splits):
            for p in points:
                bis.split([1 if j == i else 0 for j in range(2)], p)
        out.append(lt.block_tensor(ctx, bis))
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    out[0].from_dense(a)
    out[1].from_dense(b)
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 0)
    op = lt.btod_contract2(con, out[0], out[1])
    if tile is not None:
        op.set_tile(tile)
    return op, out[2], a @ b, 2 * (k + 2) * EPS * (abs(a) @ abs(b))


def _merged(ctx, reqs, add=False, d=1.0):
    """All requests behind a medium one, so that they are ready together."""
    big = _operation(ctx, 3000, 3000, 1500, 99, 19)
    srv = lt.server(ctx, 64)
    try:
        t = [srv.submit(big[0], big[1])] + [srv.submit(r[0], r[1], add, d) for r in reqs]
        for x in t:
            assert srv.wait(x)["status"] == 0
    finally:
        srv.close()


# 2 m n k just below and above 5e7
@pytest.mark.parametrize("m,n,k,tile", [(77, 65, 4900, 14), (77, 65, 5100, 19), (130, 100, 1900, 14), (130, 100, 1950, 19)])
def test_tile_by_flops(gpu_ctx, m, n, k, tile):
    reqs = [_operation(gpu_ctx, m, n, k, s) for s in range(4)]
    _merged(gpu_ctx, reqs)
    for op, c, ref, bound in reqs:
        assert op.stats()["tile_cfg"] == tile
        assert np.all(abs(c.to_dense() - ref) <= bound)
    _merged(gpu_ctx, reqs, True, 0.5)
    for op, c, ref, bound in reqs:
        assert op.stats()["tile_cfg"] == tile
        assert np.all(abs(c.to_dense() - 1.5 * ref) <= 2 * bound)


@pytest.mark.parametrize("tile", [4, 13, 23, 24, 25, 14, 19, 26])
def test_merged_equals_alone(gpu_ctx, tile):
    reqs = [_operation(gpu_ctx, *shape, s, tile) for s, shape in enumerate([(77, 65, 2500), (130, 100, 1900), (50, 33, 5000), (17, 129, 40)])]
    _merged(gpu_ctx, reqs)
    got = [r[1].to_dense() for r in reqs]
    for (op, c, ref, bound), x in zip(reqs, got):
        assert np.all(abs(x - ref) <= bound)
        op.perform(c)
        assert np.array_equal(c.to_dense(), x)


def test_sliced_equals_alone(gpu_ctx):
    """A request beyond 2e11 FLOPs runs in slices; its tiles (900 of 64 x 64)
    are cut along k, the parts' sums added after the last slice."""
    m, n, k = 1900, 1890, 28200
    op, c, a, b = _large(gpu_ctx, m, n, k)
    op.set_tile(19)
    srv = lt.server(gpu_ctx)
    try:
        assert srv.wait(srv.submit(op, c))["status"] == 0
    finally:
        srv.close()
    got = c.to_dense()
    op.perform(c)
    assert np.array_equal(c.to_dense(), got)
    rows = slice(0, m, 97)
    assert np.all(abs(got[rows] - a[rows] @ b) <= 2 * (k + 2) * EPS * (abs(a[rows]) @ abs(b)))


def _large(ctx, m, n, k):
    rng = np.random.default_rng(8)
    a, b = rng.random((m, k)), rng.random((k, n))
    t = []
    for shape, data in (((m, k), a), ((k, n), b), ((m, n), None)):
        t.append(lt.block_tensor(ctx, lt.block_index_space(shape)))
        if data is not None:
            t[-1].from_dense(data)
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 0)
    return lt.btod_contract2(con, t[0], t[1]), t[2], a, b
