"""Grouped performs run pairs of a contraction list that are the same product
of stored blocks once, with the sum of their coefficients; the reference here
(compute_block on the host: FP64 loops over the block's full list) runs every
pair."""
import numpy as np
import pytest

import golden_cases as G
import libtensor_amd as lt
import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["ladder_full", "ladder_spin", "ladder_perm", "ladder_label", "ladder_nosym",
                                  "self_ladder", "randsym_211", "randsym_222", "rand_221"])
@pytest.mark.parametrize("mode", [lt.LT_MODE_GROUPED, lt.LT_MODE_PER_BLOCK])
def test_every_block_equals_its_full_list(gpu_ctx, name, mode):
    prob, dense, meta, result = G.load(name)
    a, b, op = P.build(gpu_ctx, prob, dense)
    c = P.make_result_tensor(gpu_ctx, prob)
    op.perform(c, mode)
    top = np.abs(result).max()
    for x in op.get_schedule():
        ref = op.compute_block_host(x, c.block_dims(x))
        assert np.abs(c.get_block(x) - ref).max() <= 1e-12 * top, x


def test_statistics_count_the_schedule(gpu_ctx):
    """FLOPs and pairs are the schedule's, whatever ran."""
    prob, dense, meta, result = G.load("ladder_full")
    a, b, op = P.build(gpu_ctx, prob, dense)
    c = P.make_result_tensor(gpu_ctx, prob)
    op.perform(c)
    pairs = flops = 0
    for x in op.get_schedule():
        size = int(np.prod(c.block_dims(x)))
        for p in op.clst(x):
            d = a.block_dims(p[0])
            pairs += 1
            flops += 2 * size * d[2] * d[3]
    st = op.stats()
    assert st["n_pairs"] == pairs and st["flops"] == flops


@pytest.mark.parametrize("name,fewer", [("ladder_nosym", False), ("ring_small", False), ("ladder_full", True), ("ladder_perm", True)])
def test_executed_flops(gpu_ctx, name, fewer):
    prob, dense, meta, result = G.load(name)
    a, b, op = P.build(gpu_ctx, prob, dense)
    op.perform(P.make_result_tensor(gpu_ctx, prob))
    run, listed = op.executed_flops(), op.stats()["flops"]
    assert 0.5 * listed <= run < listed if fewer else run == listed


def test_zero_coefficient(gpu_ctx):
    """A contraction scaled by zero writes zeros."""
    prob, dense, meta, result = G.load("ladder_full")
    a, b, op = P.build(gpu_ctx, prob, dense)
    zero = lt.btod_contract2(op.contr, a, b, kc=0.0)
    c = P.make_result_tensor(gpu_ctx, prob)
    zero.perform(c)
    assert not np.any(c.to_dense())


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("where", [0, 1])
@pytest.mark.parametrize("name", ["ladder_full", "ladder_perm", "self_ladder", "randsym_222"])
def test_non_finite_elements_reach_the_result(gpu_ctx, name, where, value):
    """An infinity or a NaN in a stored block: the same elements of C are
    infinite and NaN as in the full list's sums (pairs whose coefficients
    cancel are not left out)."""
    prob, dense, meta, result = G.load(name)
    a, b, op = P.build(gpu_ctx, prob, dense)
    t = b if where else a
    x = t.req_nonzero_blocks()[0]
    blk = t.get_block(x)
    blk.flat[blk.size // 2] = value
    t.set_block(x, blk)
    c = P.make_result_tensor(gpu_ctx, prob)
    op.perform(c)
    seen = 0
    for x in op.get_schedule():
        got, ref = c.get_block(x), op.compute_block_host(x, c.block_dims(x))
        assert np.array_equal(np.isnan(got), np.isnan(ref)), x
        assert np.array_equal(np.isinf(got), np.isinf(ref)), x
        seen += np.count_nonzero(~np.isfinite(ref))
    assert seen
