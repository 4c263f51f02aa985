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


def test_cutoff_near_its_end(ctx):  # noqa: F811
    """Pairs up to the cutoff radius itself, one function G1 = fc(r): never negative, 0 at r = rc, and
    close to the exact value: cos x within 5e-16 (halved, and half an ulp for the sum with 1), its
    derivative through sin x within 6e-16 (three roundings on top)."""
    L = np.longdouble
    pi = L("3.14159265358979323846264338327950288")
    dims = [1, 1]
    for rc in (RC, 7.3, 9.0):
        u = np.nextafter(rc, np.inf) - rc
        r = np.concatenate([rc - u * np.arange(40), rc - u * 2.0 ** np.arange(6, 48),
                            rc * np.random.default_rng(3).uniform(0.05, 1.0, 900)])
        p = np.array([[1.0, 0.0, 0.0, 0.0]])  # E = G1
        g = fa.GFunctions([1], [rc])
        ctx.upload_model(fa.Netstat(g, [14], dims, 0, p))
        b = ctx.batch([fa.Geometry([[0.0, 0.0, 0.0], [x, 0.0, 0.0]], [14] * 2, [0] * 2) for x in r],
                      fa.FNET_FP64)
        G, F = b.acsf()[::2, 0], b.forces()[1::2, 0]
        b.close()
        x = pi * r.astype(L) / L(rc)
        fc, dfc = (np.cos(x) + 1) / 2, -np.sin(x) * pi / (2 * L(rc))
        print("rc", rc, "fc", float(np.abs(G - fc).max()), "min", G.min(),
              "sin", float(np.abs(F + 2 * dfc).max() * L(rc) / pi), flush=True)
        assert (G >= 0.0).all() and (G[r == rc] == 0.0).all() and (r == rc).any()
        assert np.abs(G - fc).max() <= 0.5 * 5e-16 + 1.2e-16
        assert np.abs(F + 2 * dfc).max() * L(rc) / pi <= 6e-16 + 3 * 1.2e-16  # both atoms' energies
