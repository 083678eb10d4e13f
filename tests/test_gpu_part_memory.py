"""Memory for the partial sums of tiles cut along k: bounded by the grouped
launch's tiles whatever the number of C blocks, and no part of what a plan, a
batch or a request must fit."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53
M, N, K = 96, 128, 16000            # 96 C blocks of one row that share B


@pytest.fixture(scope="module")
def operands():
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    return a, b, a @ b, 2 * (K + 2) * EPS * (abs(a) @ abs(b))


def _tensor(ctx, dims, points, data=None):
    bis = lt.block_index_space(dims)
    for p in points:
        bis.split([1, 0], p)
    t = lt.block_tensor(ctx, bis)
    if data is not None:
        t.from_dense(data)
    return t


def _op(ctx, a, b, tile):
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 0)
    op = lt.btod_contract2(con, _tensor(ctx, a.shape, range(1, M), a), _tensor(ctx, b.shape, [], b))
    if tile is not None:
        op.set_tile(tile)
    return op, _tensor(ctx, (M, N), range(1, M))


@pytest.fixture
def ctx():
    c = lt.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("tile", [19, 26, None])
def test_bounded_by_the_grouped_launch(ctx, operands, tile):
    a, b, ref, bound = operands
    op, c = _op(ctx, a, b, tile)
    op.perform(c)                                     # also makes C's memory
    op.close()
    op, c2 = _op(ctx, a, b, tile)
    used = ctx.mem()[0]
    op.perform(c)
    first = c.to_dense()
    assert np.all(abs(first - ref) <= bound)
    # below 1536 places of at most 96 x 128, and the plan's lists
    assert ctx.mem()[0] - used < 1536 * 96 * 128 * 8 + (64 << 20)
    used = ctx.mem()[0]
    op.perform(c, lt.LT_MODE_PER_BLOCK)
    assert ctx.mem()[0] - used < 4 * 1536 * 96 * 128 * 8
    if tile is not None:
        assert np.array_equal(c.to_dense(), first)
    op.perform(c)
    assert np.array_equal(c.to_dense(), first)


@pytest.mark.parametrize("tile", [19, 26])
@pytest.mark.parametrize("mode", [lt.LT_MODE_GROUPED, lt.LT_MODE_PER_BLOCK])
def test_without_room_the_tiles_run_whole(ctx, operands, tile, mode):
    a, b, ref, bound = operands
    op, c = _op(ctx, a, b, tile)
    op.perform(c)
    op.close()
    op, c2 = _op(ctx, a, b, tile)
    # room for the lists (24 bytes per C block row, 32 per row of an A block), not for partial sums
    ctx.set_cap(ctx.mem()[0] + (1 << 20))
    op.perform(c, mode)
    assert op.stats()["n_batches"] == 1
    assert np.all(abs(c.to_dense() - ref) <= bound)
    op.perform_add(c, 0.5, mode)
    assert op.stats()["n_batches"] == 1
    assert np.all(abs(c.to_dense() - 1.5 * ref) <= 2 * bound)


@pytest.mark.parametrize("tile", [19, 26])
@pytest.mark.parametrize("room", [1 << 20, 1 << 30])
def test_requests(ctx, operands, tile, room):
    """Two requests in one batch, whose tiles are cut where there is room."""
    a, b, ref, bound = operands
    ops = [_op(ctx, a, b, tile) for _ in range(3)]
    alone = ops[2][1]
    for op, c in ops:
        op.perform(c)
        op.close()
    expect = alone.to_dense()
    ops = [(_op(ctx, a, b, tile)[0], c) for _, c in ops]
    ctx.set_cap(ctx.mem()[0] + room)
    srv = lt.server(ctx, max_batch=8)
    try:
        for rep in range(2):
            for st in [srv.wait(t) for t in [srv.submit(op, c) for op, c in ops[:2]]]:
                assert st["status"] == 0, st
            for op, c in ops[:2]:
                assert np.all(abs(c.to_dense() - ref) <= bound)
                if room > (1 << 20):
                    assert np.array_equal(c.to_dense(), expect)
    finally:
        srv.close()
