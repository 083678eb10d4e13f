"""Dense calls in a context whose memory budget leaves a few KiB: the workspace
that they use where there is room is no reason to refuse them."""
import numpy as np
import pytest

import libtensor_amd as lt

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


@pytest.fixture
def ctx():
    c = lt.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("m,n,k", [(16, 64, 5000), (40, 130, 3000)])
def test_contraction_cut_along_k(ctx, m, n, k):
    rng = np.random.default_rng(m)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    da, db = lt.device_array(ctx, a.shape, a), lt.device_array(ctx, b.shape, b)
    dc = lt.device_array(ctx, (m, n))
    con = lt.contraction2(1, 1, 1)
    con.contract(1, 0)
    bound = 2 * (k + 2) * EPS * (abs(a) @ abs(b))
    ctx.set_cap(ctx.mem()[0] + (1 << 14))
    lt.tod_contract2(con, da, db, dc)
    assert np.all(abs(dc.download() - a @ b) <= bound)
    ctx.set_cap(ctx.mem()[0] + (1 << 24))
    lt.tod_contract2(con, da, db, dc, zero=False)
    assert np.all(abs(dc.download() - 2 * (a @ b)) <= 3 * bound)


def test_scalar_product(ctx):
    x = np.random.default_rng(1).standard_normal((40, 60))
    d = lt.device_array(ctx, x.shape, x)
    ctx.set_cap(ctx.mem()[0] + (1 << 13))
    assert abs(lt.tod_dotprod(d, d) - np.vdot(x, x)) <= 2 * x.size * EPS * np.vdot(x, x)
