"""Precision of the powers of a real-step progression in FP64.

Trimers whose cosine is the rounded quotient of two integers and whose other factors are common to
all functions of the group: the ratio of a value to the first member's is P^(k s), P = 1 + lambda c,
with one rounding for each of k steps, the member's own and those of the two values' scale and sum
(six): (k + 6) half ulps, however P's own rounding would grow in the power.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_workloads import ctx  # noqa: F401

pytestmark = pytest.mark.gpu
L = np.longdouble


def _trimers():
    out, cos = [], []
    for m in range(2, 24):
        for n in range(1, m):
            x, y, h = m * m - n * n, 2 * m * n, m * m + n * n
            for sx in (1.0, -1.0):
                q = 2.0 ** 8
                out.append(fa.Geometry([[0.0, 0.0, 0.0], [h * q, 0.0, 0.0], [sx * x * q, y * q, 0.0]],
                                       [14, 1, 8], [2, 0, 1]))
                cos.append(sx * x / h)
    return out, np.array(cos)


@pytest.mark.parametrize("x0,s,n", [(1.0, 15.0 / 7.0, 8), (1.25, 2.3, 8), (1.5, 0.75, 3), (1.0, 1.5, 4)])
def test_ratio_of_members(ctx, x0, s, n):  # noqa: F811
    print("progression", x0, s, n, flush=True)
    geos, c = _trimers()
    xi = np.array([x0 + k * s for k in range(n) for _ in (0, 1)])
    lam = np.array([1.0, -1.0] * n)
    f = 2 * n
    g = fa.GFunctions([5] * f, [2.0 ** 20] * f, eta=[0.0] * f, xi=xi, lam=lam, z1=[1] * f, z2=[8] * f)
    dims = [f, 2, 1]
    ctx.upload_model(fa.Netstat(g, [1, 8, 14], dims, 0, W.random_params(dims, 3, 1)))
    b = ctx.batch(geos, fa.FNET_FP64)
    G = b.acsf()[::3].astype(L)
    b.close()
    u = np.finfo(np.float64).eps / 2
    for l in (0, 1):
        P = 1 + L(lam[l]) * c.astype(L)
        for k in range(1, n):
            d = L(xi[2 * k]) - L(xi[0])
            want = np.exp(d * np.log(P / 2))
            err = np.abs(G[:, 2 * k + l] / G[:, l] / want - 1)
            print("lambda %+d xi %.3f: error %.2g, rms %.2g" %
                  (lam[l], xi[2 * k], err.max(), np.sqrt((err * err).mean())), flush=True)
            assert err.max() <= (k + 6) * u
