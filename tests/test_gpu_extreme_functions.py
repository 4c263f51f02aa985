"""Function parameters at the ends of their range, against the FP64 oracle (1e-10 of the largest
value in FP64, 1e-5 in FP32): exponents so large that every exponential vanishes."""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_workloads import _clusters, _oracle_all, ctx  # noqa: F401

pytestmark = pytest.mark.gpu
RC = 6.0 * fa.AA__BOHR


def _features(ctx, geos, g, mode):  # noqa: F811
    dims = [len(g), 3, 1]
    ns = fa.Netstat(g, [1, 8], dims, 0, W.random_params(dims, 2, 9))
    ctx.upload_model(ns)
    b = ctx.batch(geos, mode)
    G, F = b.acsf(), b.forces()
    b.close()
    return ns, G, F


@pytest.mark.parametrize("mode,eta", [(fa.FNET_FP64, e) for e in (1e3, 1e20, 1e42, 1e300, np.inf)] +
                         [(fa.FNET_FP32, e) for e in (1e3, 1e20)])
def test_vanishing_exponentials(ctx, mode, eta):  # noqa: F811
    print("eta", eta, "mode", mode, flush=True)
    geos = _clusters(4)
    g = fa.GFunctions([2, 2, 5, 5], [RC] * 4, eta=[0.01, eta, 0.01, eta], rs=[0.0] * 4,
                      xi=[0.0, 0.0, 4.0, 4.0], lam=[0.0, 0.0, 1.0, 1.0])
    ns, G, F = _features(ctx, geos, g, mode)
    G0 = _oracle_all(geos, ns)[0]
    assert np.isfinite(G0).all() and (G0[:, [1, 3]] == 0.0).all()
    assert np.abs(G - G0).max() <= (1e-10 if mode == fa.FNET_FP64 else 1e-5) * np.abs(G0).max()
    if eta < 1e100:  # (the derivative's eta r overflows beyond)
        assert np.isfinite(F).all()
