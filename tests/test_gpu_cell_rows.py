"""Rows of the cell-list search around its capacities: hits are put in the reference's order by ranks
up to 256 slots, by a sorting network beyond.  Random cells of 21 A with a 5 A cutoff (4 bins per
axis) and about 4, 64, 128, 200 and 300 neighbours per atom: the counted list and the one-pass list
must be the oracle's rows exactly, entry by entry."""
import numpy as np
import pytest

import fortnet_amd as fa
from test_gpu_neighbours import _check_rows, _model, ctx  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("atoms", [64, 1080, 1150, 2250, 3550, 5300])
def test_rows_in_reference_order(ctx, atoms):  # noqa: F811
    A = fa.AA__BOHR
    rc, lat = 5.0 * A, np.diag([21.0, 21.5, 22.0]) * A
    rng = np.random.default_rng(atoms)
    xyz = rng.uniform(-0.2, 1.2, size=(atoms, 3)) @ lat
    geo = fa.Geometry(xyz, [14] * atoms, [0] * atoms, lat)
    ctx.upload_model(_model(rc))
    for prec in (fa.FNET_FP64, fa.FNET_FP32):
        b = ctx.batch([geo], prec)
        for k in range(2):
            b.neighbour_list()
            rp, j, img = b.neighbours()
            if k == 0:
                print("atoms", atoms, "longest row", np.diff(rp).max(), flush=True)
            if prec == fa.FNET_FP64:
                _check_rows([geo], rc, rp, j, img)
                want = rp, j, img
            else:
                assert all(np.array_equal(x, y) for x, y in zip((rp, j, img), want))
        b.close()
