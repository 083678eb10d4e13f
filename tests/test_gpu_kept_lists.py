"""Descriptor lists kept between calls: an iteration's many scalar products
leave those of its sums in place, they are bounded, and given back where
device memory runs short."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    c = lt.Context(0)
    yield c
    c.close()


def _tensor(ctx, dims, parts):
    bis = lt.block_index_space(dims)
    for i, d in enumerate(dims):
        for p in range(1, parts):
            bis.split([1 if j == i else 0 for j in range(len(dims))], p * d // parts)
    t = lt.block_tensor(ctx, bis)
    t.random(sum(dims))
    return t


def _sum(ctx):
    x, y = (_tensor(ctx, (24, 24, 24), 12) for _ in range(2))     # 1728 blocks
    r = _tensor(ctx, (24, 24, 24), 12)
    add = lambda: lt.btod_add([(x, None, 0.5), (y, (2, 1, 0), 2.0)], r)
    add()
    return add, r, 0.5 * x.to_dense() + 2.0 * y.to_dense().transpose(2, 1, 0)


def test_scalar_products_beside_sums(ctx):
    add, r, ref = _sum(ctx)
    v = [_tensor(ctx, (3, 4), 1) for _ in range(9)]
    dense = [t.to_dense() for t in v]
    lt.tod_dotprod(*[lt.device_array(ctx, (4,), np.ones(4))] * 2)     # makes the staging area
    used = ctx.mem()[0]
    for rep in range(2):
        for i in range(9):
            for j in range(9):
                d = lt.btod_dotprod(v[i], v[j])
                assert abs(d - np.vdot(dense[i], dense[j])) <= 24 * 2.0 ** -53 * np.vdot(abs(dense[i]), abs(dense[j]))
    # the sum's lists are there still (beside at most 64 short ones)
    assert used <= ctx.mem()[0] <= used + 64 * 4096
    add()
    assert np.allclose(r.to_dense(), ref, rtol=1e-15, atol=1e-15)


def test_given_back_when_memory_runs_short(ctx):
    used0 = ctx.mem()[0]
    add, r, ref = _sum(ctx)
    kept = ctx.mem()[0]
    ctx.set_cap(kept + 4096)
    a = lt.device_array(ctx, (8192,))                            # 64 KiB: less than the lists
    assert ctx.mem()[0] <= kept + 4096
    a.free()
    add()
    assert np.allclose(r.to_dense(), ref, rtol=1e-15, atol=1e-15)
