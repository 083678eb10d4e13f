"""Workgroup-tiled GEMM kernels at the edges of their tiles: matrix products
whose extents sit around the 16-row fragments, 64-column tiles and 16-k
chunks, in every operand layout, one block or several (stacked C blocks,
several pairs of ragged extents per C block)."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

WG = [14, 15, 16, 17, 19, 20, 21, 26, 27]


def _tensor(ctx, dims, splits):
    bis = lt.block_index_space(dims)
    for d, points in enumerate(splits):
        for p in points:
            bis.split([1 if i == d else 0 for i in range(len(dims))], p)
    return lt.block_tensor(ctx, bis)


def _product(ctx, m, n, k, ta, tb, sm, sn, sk, seed):
    rng = np.random.default_rng(seed)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    ta_, tb_ = (a.T if ta else a), (b.T if tb else b)
    bta = _tensor(ctx, ta_.shape, (sk, sm) if ta else (sm, sk))
    btb = _tensor(ctx, tb_.shape, (sn, sk) if tb else (sk, sn))
    bta.from_dense(ta_)
    btb.from_dense(tb_)
    c = lt.contraction2(1, 1, 1)
    c.contract(0 if ta else 1, 1 if tb else 0)
    return a, b, lt.btod_contract2(c, bta, btb, kc=0.5), _tensor(ctx, (m, n), (sm, sn))


SHAPES = [(1, 1, 1), (16, 64, 16), (17, 65, 17), (15, 63, 15), (33, 1, 31), (1, 129, 64), (113, 66, 47),
          (112, 128, 33), (97, 64, 100), (80, 70, 5), (81, 191, 257)]


@pytest.mark.parametrize("cfg", WG)
@pytest.mark.parametrize("layout", [(False, False), (True, False), (False, True), (True, True)])
def test_tile_edges(gpu_ctx, cfg, layout):
    ta, tb = layout
    for m, n, k in SHAPES:
        for split in (False, True):
            sm = [m // 3, m // 3 + 1] if split and m > 5 else []
            sn = [n // 2] if split and n > 5 else []
            sk = [k // 4, k // 4 + 1, k - 2] if split and k > 12 else []
            a, b, op, c = _product(gpu_ctx, m, n, k, ta, tb, sm, sn, sk, m * 7919 + n * 31 + k)
            op.set_tile(cfg)
            op.perform(c, lt.LT_MODE_GROUPED)
            got = c.to_dense()
            # |error| of a length-k FP64 sum in any order: at most
            # (k + 2) u sum |a| |b|, u = 2^-53 (N. Higham, Accuracy and
            # Stability of Numerical Algorithms, 3.1)
            bound = (k + 2) * 2.0 ** -53 * (np.abs(a) @ np.abs(b)) * 2
            assert np.all(np.abs(got - 0.5 * (a @ b)) <= bound), (m, n, k, split)
            op.perform(c, lt.LT_MODE_PER_BLOCK)
            assert np.array_equal(c.to_dense(), got), (m, n, k, split)


@pytest.mark.parametrize("cfg", WG)
def test_non_finite_values_stay_in_their_rows_and_columns(gpu_ctx, cfg):
    """An infinity or a NaN in the last k of a ragged extent reaches its own row
    or column only (the zeros past the extent are set, not multiplied)."""
    a, b, op, c = _product(gpu_ctx, 20, 70, 19, False, False, [], [], [], 5)
    a[3, 18] = np.inf
    b[18, 66] = np.nan
    op.a.from_dense(a)
    op.b.from_dense(b)
    op.set_tile(cfg)
    op.perform(c, lt.LT_MODE_GROUPED)
    got = c.to_dense()
    with np.errstate(invalid="ignore"):
        ref = 0.5 * (a @ b)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    assert np.array_equal(np.isnan(got), np.isnan(ref))


# 24 chunks of k and more: the tiles are cut into parts, inside pairs and at
# their ends, and a second kernel adds the parts' sums
CUT = [(33, 70, 400), (16, 64, 3000), (97, 129, 1033), (113, 66, 777)]


@pytest.mark.parametrize("cfg", WG)
@pytest.mark.parametrize("layout", [(False, False), (True, False), (False, True), (True, True)])
def test_tiles_cut_along_k(gpu_ctx, cfg, layout):
    ta, tb = layout
    for m, n, k in CUT:
        for sk in ([], [k // 2], [k // 3, k // 3 + 1, k - 17], [16 * (k // 32)]):
            print("cut tiles", cfg, layout, m, n, k, sk, flush=True)
            a, b, op, c = _product(gpu_ctx, m, n, k, ta, tb, [m // 3, m // 3 + 1], [n // 2], sk, m * 7919 + n * 31 + k)
            op.set_tile(cfg)
            ref, bound = 0.5 * (a @ b), (k + 2) * 2.0 ** -53 * (np.abs(a) @ np.abs(b)) * 2
            op.perform(c, lt.LT_MODE_GROUPED)
            got = c.to_dense()
            assert np.all(np.abs(got - ref) <= bound), (m, n, k, sk)
            op.perform(c, lt.LT_MODE_PER_BLOCK)
            assert np.array_equal(c.to_dense(), got), (m, n, k, sk)
            op.perform_add(c, -3.0, lt.LT_MODE_GROUPED)
            assert np.all(np.abs(c.to_dense() + 2 * ref) <= 5 * bound), (m, n, k, sk)
            op.perform_add(c, 3.0, lt.LT_MODE_PER_BLOCK)
            assert np.all(np.abs(c.to_dense() - ref) <= 9 * bound), (m, n, k, sk)
