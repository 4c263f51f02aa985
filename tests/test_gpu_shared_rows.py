"""Direct neighbour search with four waves to an atom (small batches) and one (the counted list, and
batches of more than 1024 atoms): candidate counts around multiples of 64 and 256, cells shorter
than the cutoff with hundreds of images, empty rows, and batches on both sides of the line must give
the oracle's rows exactly, entry by entry, in both precisions."""
import numpy as np
import pytest

import fortnet_amd as fa
from test_gpu_neighbours import _check_rows, _model, ctx  # noqa: F401

pytestmark = pytest.mark.gpu
A = fa.AA__BOHR


def _cluster(n, seed, size):
    rng = np.random.default_rng(seed)
    return fa.Geometry(rng.uniform(0, size, (n, 3)) * A, [14] * n, [0] * n)


def _cell(n, seed, size):
    rng = np.random.default_rng(seed)
    lat = (np.diag([size, 1.1 * size, 0.9 * size]) + 0.1 * rng.normal(size=(3, 3))) * A
    return fa.Geometry(rng.uniform(-0.3, 1.3, (n, 3)) @ lat, [14] * n, [0] * n, lat)


SETS = {
    "one": lambda: [_cluster(1, 1, 1.0)],
    "steps": lambda: [_cluster(n, n, 9.0) for n in (2, 64, 65, 66, 129, 257, 258)],
    "images": lambda: [_cell(1, 3, 2.2), _cell(2, 4, 2.9), _cell(5, 5, 3.4), _cell(31, 6, 7.0),
                       _cluster(3, 7, 30.0)],
    "at_line": lambda: [_cell(64, 10 + k, 10.0) for k in range(16)],
    "past_line": lambda: [_cell(64, 10 + k, 10.0) for k in range(16)] + [_cluster(1, 9, 1.0)],
}


@pytest.mark.parametrize("name", sorted(SETS))
def test_shared_rows(ctx, name):  # noqa: F811
    geos = SETS[name]()
    print("rows", name, [g.n for g in geos], flush=True)
    rc = 5.0 * A
    ctx.upload_model(_model(rc))
    for prec in (fa.FNET_FP64, fa.FNET_FP32):
        b = ctx.batch(geos, prec)
        for k in range(2):  # counted, then in one pass into the kept rows
            b.neighbour_list()
            rp, j, img = b.neighbours()
            if prec == fa.FNET_FP64:
                _check_rows(geos, rc, rp, j, img)
                want = rp, j, img
            else:
                assert all(np.array_equal(x, y) for x, y in zip((rp, j, img), want))
        b.close()
