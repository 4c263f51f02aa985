"""Lists built with the capacities of the list before, without a read-back, by each call that asks for
results: when a row has outgrown the ACSF slice, or the row capacity, what the call returns is computed
again on a list of the right size.  Results equal a fresh batch's, bit for bit.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_neighbours import ctx  # noqa: F401

pytestmark = pytest.mark.gpu
RC = 5.0 * fa.AA__BOHR


def _model():
    g = fa.GFunctions.concat([fa.GFunctions([2] * 2, [RC] * 2, eta=[0.1, 0.02]),
                              fa.GFunctions([5] * 2, [RC] * 2, eta=[0.02] * 2, xi=[1, 4], lam=[1.0, -1.0])])
    dims = [len(g), 6, 1]
    return fa.Netstat(g, [14], dims, 0, W.random_params(dims, 1, 3), np.full(len(g), 2.0),
                      np.full(len(g), 3.0))


def _energy_forces(b):
    return [*b.energy(), b.forces()]


def _train(b):
    grad, pred = b.train_gradients(np.arange(b.S, dtype=float)[:, None])
    return [grad, pred, np.array([b.loss])]


CALLS = {"acsf": lambda b: [b.acsf()], "energy": lambda b: list(b.energy()),
         "forces": lambda b: [b.forces()], "energy_forces": _energy_forces,
         "forces_energy": lambda b: [b.forces(), *b.energy()], "train": _train,
         "acsf_train": lambda b: [b.acsf()] + _train(b)}


def _longest(ctx, geos):  # noqa: F811
    b = ctx.batch(geos, fa.FNET_FP64)
    b.neighbour_list()
    rp = b.neighbours()[0]
    b.close()
    return int(np.diff(rp).max())


def _scaled(geos, f):
    return [fa.Geometry(g.coords * f, g.atnum, g.species, g.latvecs * f) for g in geos]


@pytest.mark.parametrize("precision", [fa.FNET_FP64, fa.FNET_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("cells", [[2] * 3, [2] * 140, [6, 2]], ids=["pinned", "copied", "bins"])
@pytest.mark.parametrize("call", sorted(CALLS))
def test_outgrown_rows(ctx, call, cells, precision):  # noqa: F811
    ctx.upload_model(_model())
    geos = [W.si_diamond(n, n, n, 0.1, 50 + k) for k, n in enumerate(cells)]
    m0 = _longest(ctx, geos)
    slice0, cap0 = (m0 + 7) // 8 * 8, (m0 + m0 // 4 + 8 + 7) // 8 * 8
    fn = CALLS[call]
    for what in ("slice", "capacity"):
        for f in np.arange(0.99, 0.7, -0.01):  # compressed until the rows outgrow it
            dense = _scaled(geos, f)
            m1 = _longest(ctx, dense)
            if m1 > (slice0 if what == "slice" else cap0):
                break
        print(call, cells[:2], precision, what, "rows", m0, "->", m1, "slice", slice0, "capacity", cap0,
              flush=True)
        assert slice0 < m1 <= cap0 if what == "slice" else m1 > cap0
        ref = ctx.batch(dense, precision)
        want = fn(ref)
        ref.close()
        b = ctx.batch(geos, precision)
        first = fn(b)  # the counted list, whose capacities the next one takes
        xyz = [np.concatenate([g.coords for g in q]) for q in (geos, dense)]
        lat = [np.stack([g.latvecs for g in q]) for q in (geos, dense)]
        for turn in range(2):
            b.update_coords(xyz[1], lat[1])
            got = fn(b)
            assert len(got) == len(want) and all(np.array_equal(x, y) for x, y in zip(got, want))
            b.update_coords(xyz[0], lat[0])
            got = fn(b)
            assert all(np.array_equal(x, y) for x, y in zip(got, first))
        b.close()


@pytest.mark.parametrize("n", [5, 97, 210])
def test_staged_copies_of_two_batches(ctx, n):  # noqa: F811
    """Coordinates staged for one batch, then more than the ring holds for another, without a result
    read between them: neither overwrites the other's.  n sets where the ring's end falls."""
    ctx.upload_model(_model())
    rng = np.random.default_rng(n)
    ga = [W.si_diamond(2, 2, 2, 0.1, k) for k in range(7)]
    gb = [W.si_diamond(2, 2, 2, 0.1, 100 + k) for k in range(n)]
    xs = []
    for geos in (ga, gb):
        x0 = np.concatenate([g.coords for g in geos])
        xs.append([x0 + 0.05 * rng.normal(size=x0.shape) for _ in range(2)])
    want = []
    for geos, x in zip((ga, gb), xs):
        want.append([])
        for v in x:
            b = ctx.batch(geos, fa.FNET_FP64)
            b.update_coords(v)
            want[-1].append(b.acsf())
            b.close()
    a, b = ctx.batch(ga, fa.FNET_FP64), ctx.batch(gb, fa.FNET_FP64)
    a.acsf()
    b.acsf()
    rounds = 1 + (3 << 20) // (24 * 64 * n)
    for turn in range(2):
        for k in range(2):
            a.update_coords(xs[0][k])
            for r in range(rounds):
                b.update_coords(xs[1][(r + k) % 2])
                if turn and r % 5 == 0:
                    a.update_coords(xs[0][k])
            assert np.array_equal(a.acsf(), want[0][k])
            assert np.array_equal(b.acsf(), want[1][(rounds - 1 + k) % 2])
    a.close()
    b.close()
