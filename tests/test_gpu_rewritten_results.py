"""Copies and sums into a tensor that the same call wrote before: its structure
version is kept, so operations that read it keep their plans, unless its
blocks or symmetry changed in between."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

DIMS, POINTS = (10, 12), ([3], [5, 8])


def _tensor(ctx, sym=None, data=None, dims=DIMS, points=POINTS):
    bis = lt.block_index_space(dims)
    if dims[0] == dims[1]:
        for p in points[0]:
            bis.split([1, 1], p)
    else:
        for i in range(2):
            for p in points[i]:
                bis.split([int(j == i) for j in range(2)], p)
    t = lt.block_tensor(ctx, bis)
    if sym is not None:
        t.insert(sym)
    if data is not None:
        t.from_dense(data)
    return t


def _calls(ctx, rng):
    x, y = (rng.standard_normal(DIMS) for _ in range(2))
    a, b = _tensor(ctx, data=x), _tensor(ctx, data=y)
    return {"copy": (lambda r: lt.btod_copy(a, r, None, -2.0), a, lambda: -2.0 * a.to_dense()),
            "add": (lambda r: lt.btod_add([(a, None, 0.5), (b, None, 4.0)], r), a,
                    lambda: 0.5 * a.to_dense() + 4.0 * b.to_dense())}


@pytest.mark.parametrize("kind", ["copy", "add"])
def test_structure_kept_and_changed(gpu_ctx, kind):
    call, a, ref = _calls(gpu_ctx, np.random.default_rng(1))[kind]
    r = _tensor(gpu_ctx)
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 1)
    call(r)
    op = lt.btod_contract2(con, r, r)
    c = _tensor(gpu_ctx, dims=(10, 10), points=([3], [3]))

    def check():
        call(r)
        op2 = lt.btod_contract2(con, r, r)
        assert np.array_equal(r.to_dense(), ref())
        op2.perform(c)
        product()

    def product():
        x = ref()
        bound = 2 * (DIMS[1] + 2) * 2.0 ** -53 * (abs(x) @ abs(x).T)     # a sum of 12 products, on both sides
        assert np.all(abs(c.to_dense() - x @ x.T) <= bound)

    call(r)
    op.perform(c)
    n = op.stats()["n_plans"]
    a.set_block(a.req_nonzero_blocks()[1], np.ones(a.block_dims(a.req_nonzero_blocks()[1])))   # data only
    call(r)
    op.perform(c)
    assert op.stats()["n_plans"] == n                      # r's version did not change
    product()
    r.zero_block(r.req_nonzero_blocks()[2])                # a block gone
    check()
    r.zero()
    check()
    x = a.req_nonzero_blocks()[0]                          # an operand's block gone: r's must go with it
    a.zero_block(x)
    check()
    a.set_block(x, np.full(a.block_dims(x), 7.0))          # and back
    check()
    lt.btod_copy(a, r, None, 9.0, add=True)                # another call wrote r, structure alike
    check()


def test_symmetry_changed_between(gpu_ctx):
    """r, rewritten by the same sum, was given another symmetry by another call."""
    rng = np.random.default_rng(2)
    s = rng.standard_normal((9, 9))
    n = rng.standard_normal((9, 9))
    sym = _tensor(gpu_ctx, lt.se_perm((1, 0), 1.0), s + s.T, (9, 9), ([4], [4]))
    plain = _tensor(gpu_ctx, None, n, (9, 9), ([4], [4]))
    r = _tensor(gpu_ctx, None, None, (9, 9), ([4], [4]))
    for i in range(3):
        lt.btod_add([(sym, None, 0.5), (sym, None, 0.25)], r)
        assert np.allclose(r.to_dense(), 0.75 * (s + s.T), rtol=1e-15, atol=1e-15)
        assert len(r.req_nonzero_blocks()) == 3
        if i == 1:
            lt.btod_add([(plain, None, 1.0), (sym, None, 1.0)], r)
            assert np.allclose(r.to_dense(), n + s + s.T, rtol=1e-15, atol=1e-15)
            assert len(r.req_nonzero_blocks()) == 4
