"""A small batch gives each centre a block of several waves (one per share of its functions); a
batch of more than a few thousand centres one wave.  One set of structures alone and beside so many
copies of itself that every number of waves occurs must give the same features, energies and
forces: the waves' shares are the same sums, and only the adjoint adds the shares' FP64 entry
gradients in another order (some eps of the largest share: 1e-12 of the largest value in FP64).  In
FP32 the kernels may also contract a product and a sum differently, one FP32 rounding per term
(6e-8): 1e-6 of the largest feature and 1e-5 of the largest force.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = fa.Context(0)
    yield c
    c.close()


def _geos(name):
    if name == "si_cells":
        return W.config(name, 0.001)[0][:2]
    if name == "ternary":
        return [W.ternary_cell(3, 16, 40), W.ternary_cell(4, 16, 40)]
    return [W.water_box(41, 9, 6.5), W.water_box(42, 1, 5.0), W.water_box(43, 12, 7.2)]


@pytest.mark.parametrize("nout", [1, 2])
@pytest.mark.parametrize("precision", [fa.FNET_FP64, fa.FNET_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", ["water", "ternary", "si_cells"])
def test_shared_centres_equal_single_waves(ctx, name, precision, nout):
    print("split centres", name, precision, nout, flush=True)
    _, ns, _ = W.config(name, 0.001)
    geos = _geos(name)
    dims = list(ns.dims[:-1]) + [nout]
    ns = fa.Netstat(ns.g, ns.species_z, dims, ns.activation, W.random_params(dims, len(ns.species_z), 5))
    ctx.upload_model(ns)
    b = ctx.batch(geos, fa.FNET_FP64)
    ns = W.with_zscore(ns, b.acsf())
    b.close()
    ctx.upload_model(ns)
    N = sum(g.n for g in geos)
    out = []
    for waves in (1, 2, 3, 5, 8):
        copies = 1 + 8192 // (waves * N) if waves == 1 else max(1, 8192 // (waves * N))
        b = ctx.batch(geos * copies, precision)
        r = [b.acsf(), b.energy()[1], b.forces()]
        b.close()
        out.append([x[:N] for x in r])
        for x in r:  # every copy like the first
            assert np.array_equal(x[-N:], x[:N])
    tol = (1e-13, 1e-12, 1e-12) if precision == fa.FNET_FP64 else (1e-6, 1e-5, 1e-5)
    for r in out[1:]:
        for x, x0, t in zip(r, out[0], tol):
            assert np.abs(x - x0).max() <= t * max(1.0, np.abs(x0).max())
