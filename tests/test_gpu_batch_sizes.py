"""One set of small cells (1, 15, 16 and 17 atoms) at the head of batches on either side of every line
that a batch's size draws: networks whose waves share 16 atoms or run 16 each (2560 parts), results
written to pinned memory or copied (8192 outputs), the mirror search beside the networks or on its
own stream (24 576 atoms), arrays staged through the pinned ring or copied on their own (512 KB).
Each of these keeps the sums and their order, so the set's energies and forces must be the same
bits; layer widths cover one to four output blocks of a wave.  Repeated uploads run the ring around
several times.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_neighbours import _model, ctx  # noqa: F401

pytestmark = pytest.mark.gpu
A = fa.AA__BOHR


def _cells():
    out = []
    for k, n in enumerate((1, 15, 16, 17)):
        rng = np.random.default_rng(70 + k)
        lat = np.diag([2.4, 2.6, 2.5]) * n ** (1.0 / 3.0) * A
        sp = rng.integers(0, 2, n)
        out.append(fa.Geometry(rng.uniform(0, 1, (n, 3)) @ lat, np.array([6, 14])[sp], sp, lat))
    return out


@pytest.mark.parametrize("precision", [fa.FNET_FP32, fa.FNET_BF16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("widths", [[25, 1], [64, 64, 1], [65, 1], [128, 128, 1], [40, 250, 1]])
def test_same_bits_at_every_size(ctx, widths, precision):  # noqa: F811
    cells = _cells()
    n0 = sum(g.n for g in cells)
    assert n0 == 49
    rc = 4.0 * A
    g = fa.GFunctions([2] * 6, [rc] * 6, eta=W.eta_bohr(W.log_eta(0.05, 1.5, 6)))
    dims = [6] + widths
    ns = fa.Netstat(g, [6, 14], dims, 0, W.random_params(dims, 2, 3), np.full(6, 0.5),
                    np.full(6, 2.0))
    ctx.upload_model(ns)
    ref = None
    for atoms in (n0, 8134, 8183, 24500, 24549, 41209):
        print("atoms", atoms, widths, precision, flush=True)
        b = ctx.batch(cells * (atoms // n0), precision)
        r = [b.energy()[1][:n0], b.forces()[:n0]]
        b.run()
        r2 = [b.energy()[1][:n0], b.forces()[:n0]]
        b.close()
        ref = ref or r
        for x, y in zip(r + r2, ref + ref):
            assert np.array_equal(x, y)


def test_repeated_uploads(ctx):  # noqa: F811
    cells = _cells() * 160  # 7840 atoms: 188 KB of coordinates a time, a 2 MB ring
    ctx.upload_model(_model(4.0 * A, (6, 14)))
    rng = np.random.default_rng(5)
    x0 = np.concatenate([g.coords for g in cells])
    b = ctx.batch(cells, fa.FNET_FP64)
    want = b.acsf()
    for k in range(40):
        b.update_coords(x0 + 0.01 * rng.normal(size=x0.shape))
        if k % 13 == 12:
            b.acsf()
    b.update_coords(x0)
    assert np.array_equal(b.acsf(), want)
    b.close()


def test_bins_by_block_or_by_kernels(ctx):  # noqa: F811
    """Bins of a structure formed by its own block, and by the kernels over all atoms that a batch
    with a structure of more than 8192 atoms takes."""
    def cell(n, size, seed):
        rng = np.random.default_rng(seed)
        lat = np.diag([size, 1.1 * size, 0.9 * size]) * A
        return fa.Geometry(rng.uniform(-0.2, 1.2, (n, 3)) @ lat, [14] * n, [0] * n, lat)

    ctx.upload_model(_model(4.0 * A))
    small, large = cell(1500, 32.0, 1), cell(8193, 55.0, 2)
    rows = []
    for geos in ([small], [small, large]):
        b = ctx.batch(geos, fa.FNET_FP64)
        b.neighbour_list()
        rp, j, img = b.neighbours()
        p = rp[small.n]
        rows.append((rp[:small.n + 1], j[:p], img[:p]))
        b.close()
    assert rows[0][1].size > 1000
    for x, y in zip(*rows):
        assert np.array_equal(x, y)
