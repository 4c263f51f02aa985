"""A resident batch under a model uploaded after it: its cells, elements and external columns are
checked against the new model as a load checks them, and its bins are laid out for the new cutoff."""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_neighbours import ctx  # noqa: F401

pytestmark = pytest.mark.gpu
A = fa.AA__BOHR


def _model(rc, species=(14,), atomid=0):
    g = fa.GFunctions([2, 2], [rc] * 2, eta=[0.1, 0.02], atomid=[atomid] * 2)
    dims = [2, 4, 1]
    return fa.Netstat(g, species, dims, 0, W.random_params(dims, len(species), 5))


@pytest.mark.parametrize("precision", [fa.FNET_FP64, fa.FNET_FP32], ids=["fp64", "fp32"])
def test_bins_follow_the_cutoff(ctx, precision):  # noqa: F811
    geos = [W.si_diamond(7, 7, 7, 0.1, 1), W.si_diamond(2, 2, 2, 0.1, 2)]
    ctx.upload_model(_model(3.5 * A))
    b = ctx.batch(geos, precision)
    b.run()
    b.energy()
    for rc in (7.0, 5.0, 3.5, 9.0):
        ctx.upload_model(_model(rc * A))
        fresh = ctx.batch(geos, precision)
        want = [fresh.energy()[1], fresh.forces(), fresh.acsf()]
        fresh.close()
        got = [b.energy()[1], b.forces(), b.acsf()]
        print("rc", rc, [float(np.abs(x - y).max()) for x, y in zip(got, want)], flush=True)
        assert all(np.array_equal(x, y) for x, y in zip(got, want))
    b.close()


def test_models_that_do_not_fit(ctx):  # noqa: F811
    """Fewer elements, external columns that the batch lacks or too large a cutoff are refused, and the
    batch is as before under the next model that fits."""
    ctx.upload_model(_model(4.0 * A, (6, 14)))
    g = W.si_diamond(2, 2, 2, 0.1, 1)
    geos = [fa.Geometry(g.coords, g.atnum, np.arange(g.n) % 2, g.latvecs)]
    b = ctx.batch(geos, fa.FNET_FP64)
    want = b.forces()
    for model, why in ((_model(4.0 * A), "species"), (_model(4.0 * A, (6, 14), 1), "external"),
                       (_model(1000.0 * A, (6, 14)), "cell too small")):
        ctx.upload_model(model)
        for call in (b.acsf, b.forces, b.run):
            with pytest.raises(fa.FnetError, match=why):
                call()
    ctx.upload_model(_model(4.0 * A, (6, 14)))
    assert np.array_equal(b.forces(), want)
    b.close()
