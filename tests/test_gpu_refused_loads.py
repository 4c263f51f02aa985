"""A batch whose reload or new cell is refused keeps the structures, tables and results that it had."""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_neighbours import ctx  # noqa: F401

pytestmark = pytest.mark.gpu
RC = 4.0 * fa.AA__BOHR


def _model():
    dims = [2, 4, 1]
    return fa.Netstat(fa.GFunctions([2, 2], [RC] * 2, eta=[0.1, 0.02]), [14], dims, 0,
                      W.random_params(dims, 1, 5))


def _huge(n=64):
    """A cell with more than 1000 bins of the cutoff along every axis: two of them are too many."""
    rng = np.random.default_rng(n)
    lat = np.diag([1002.0 * RC] * 3)
    return fa.Geometry(rng.uniform(0, 1, (n, 3)) @ lat, [14] * n, [0] * n, lat)


@pytest.mark.parametrize("when", ["before the first step", "with results"])
def test_refused_reload(ctx, when):  # noqa: F811
    ctx.upload_model(_model())
    geos = [W.si_diamond(2, 2, 2, 0.1, 1), W.si_diamond(5, 5, 5, 0.1, 2)]  # direct search and bins
    ref = ctx.batch(geos, fa.FNET_FP64)
    want = [ref.energy()[1], ref.forces()]
    ref.close()
    b = ctx.batch(geos, fa.FNET_FP64)
    if when == "with results":
        b.forces()
    bad = geos[0]
    bad = fa.Geometry(bad.coords, bad.atnum, bad.species, np.array([[1.0, 0, 0], [0, 1, 0], [1, 1, 0]]))
    for refused, why in (([_huge(), _huge()], "too many cells"), ([bad], "dependent"), ([_huge(65)] * 2, "too many")):
        with pytest.raises(fa.FnetError, match=why):
            b.reload(refused)
        assert b.N == sum(g.n for g in geos)
        assert np.array_equal(b.energy()[1], want[0]) and np.array_equal(b.forces(), want[1])
        b.update_coords(np.concatenate([g.coords for g in geos]))  # evaluated again on the old tables
        assert np.array_equal(b.energy()[1], want[0]) and np.array_equal(b.forces(), want[1])
    b.reload(geos[::-1])
    assert np.array_equal(b.forces(), np.concatenate([want[1][geos[0].n:], want[1][:geos[0].n]]))
    b.close()


def test_refused_cell(ctx):  # noqa: F811
    ctx.upload_model(_model())
    geos = [W.si_diamond(2, 2, 2, 0.1, 1), W.si_diamond(3, 3, 3, 0.1, 2)]
    coords = np.concatenate([g.coords for g in geos])
    lats = np.stack([g.latvecs for g in geos])
    b = ctx.batch(geos, fa.FNET_FP64)
    want = b.forces()
    with pytest.raises(fa.FnetError, match="too many cells"):
        b.update_coords(coords * 0.5, np.stack([np.diag([1002.0 * RC] * 3)] * 2))
    assert np.array_equal(b.forces(), want)
    b.update_coords(coords)  # the refused cells and coordinates have left nothing behind
    assert np.array_equal(b.forces(), want)
    b.close()


def test_refused_weights(ctx):  # noqa: F811
    """Datapoint weights that sum to zero are refused before the targets (here more than the staged
    copies take, so a copy command of their own) are on their way; the next call is as any other."""
    ctx.upload_model(_model())
    rng = np.random.default_rng(4)
    geos = [fa.Geometry([[0.0, 0.0, 0.0], [d, 0.0, 0.0]], [14] * 2, [0] * 2)
            for d in rng.uniform(3.0, 7.0, 35000)]
    b = ctx.batch(geos, fa.FNET_FP64)
    at, w = rng.normal(size=(b.N, 1)), rng.uniform(0.5, 1.5, b.S)
    want = b.train_gradients(a_targets=at, dp_weights=w, n_global=0)
    loss = b.loss
    with pytest.raises(fa.FnetError, match="sum to zero"):
        b.train_gradients(a_targets=np.zeros((b.N, 1)), dp_weights=np.zeros(b.S), n_global=0)
    got = b.train_gradients(a_targets=at, dp_weights=w, n_global=0)
    assert b.loss == loss and all(np.array_equal(x, y) for x, y in zip(want, got))
    b.close()
