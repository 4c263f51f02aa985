"""Exponents in steps with |lambda| > 1, where 1 + lambda cos(theta) goes below zero: its integer
powers are defined, its real ones are not (the reference's power gives NaN there), and a function
with an integer exponent must not depend on the others of its group.  Features against the FP64
oracle, 1e-10 (FP64) and 1e-5 (FP32) of the largest value, as for lambda = +-1.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_workloads import _clusters, _oracle_all, ctx  # noqa: F401

pytestmark = pytest.mark.gpu
RC = 6.0 * fa.AA__BOHR


@pytest.mark.parametrize("lams", [[1.5], [1.0, -2.5], [3.0, -1.25]])
@pytest.mark.parametrize("step", [0.5, 1.5, 3.0])
def test_large_lambda(ctx, step, lams):  # noqa: F811
    print("step", step, "lambda", lams, flush=True)
    geos = _clusters(5)
    xi = [1.0 + k * step for k in range(3) for _ in lams]
    g = fa.GFunctions.concat([fa.GFunctions.auto(RC, 3, 1),
                              fa.GFunctions([5] * len(xi), [RC] * len(xi), eta=[0.02] * len(xi),
                                            xi=xi, lam=lams * 3)])
    dims = [len(g), 4, 1]
    ns = fa.Netstat(g, [1, 8], dims, 0, W.random_params(dims, 2, 9))
    ctx.upload_model(ns)
    G0 = _oracle_all(geos, ns)[0]
    whole = np.array([ty < 4 or x == int(x) for ty, x in zip(g.type, g.xi)])
    assert np.isfinite(G0[:, whole]).all()
    for mode, tol in ((fa.FNET_FP64, 1e-10), (fa.FNET_FP32, 1e-5)):
        b = ctx.batch(geos, mode)
        G = b.acsf()
        b.close()
        assert np.abs(G - G0)[:, whole].max() <= tol * np.abs(G0[:, whole]).max()
        same = np.isnan(G0) == np.isnan(G)
        assert same.all() if mode == fa.FNET_FP64 else same[:, whole].all()
