"""A batch reloaded with no atoms after a step that left entries without a mirror.

The orphan list of the force assembly is cleared by the adjoint, which a batch without atoms does
not launch: its forces must not follow the list of the structures that were resident before.  The
pair at the cutoff of ``test_gpu_determinism`` leaves one such entry.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_determinism import _asymmetric_pair, ctx  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("launch", [fa.FNET_BATCHED, fa.FNET_PER_STRUCT], ids=["batched", "per_struct"])
@pytest.mark.parametrize("how", ["forces", "run"])
def test_no_atoms_after_orphans(ctx, how, launch):  # noqa: F811
    xi, xj, L, rc = _asymmetric_pair()
    print("asymmetric pair", xi, xj, L, rc, how, launch, flush=True)
    g = fa.GFunctions.concat([fa.GFunctions([2] * 2, [rc] * 2, eta=[0.01, 0.1]),
                              fa.GFunctions([5] * 2, [rc] * 2, eta=[0.02] * 2, xi=[1, 4],
                                            lam=[1.0, -1.0])])
    dims = [len(g), 5, 1]
    ctx.upload_model(fa.Netstat(g, [14], dims, 0, W.random_params(dims, 1, 7, scale=0.4)))
    pair = fa.Geometry([[xi, 1.0, 1.0], [xj, 1.0, 1.0], [0.5 * (xi + xj), 3.0, 1.5]], [14] * 3,
                       [0] * 3, np.diag([L, 20.0, 20.0]))
    pairs = [pair] * 40
    none = fa.Geometry([[0.0, 0.0, 0.0]], [14], [0], np.diag([L, 20.0, 20.0]))
    none.coords, none.ext = np.zeros((0, 3)), np.zeros((0, 0))  # (a structure without atoms)
    none.atnum = none.species = np.zeros(0, np.int32)
    b = ctx.batch(pairs, fa.FNET_FP64, launch)
    want = b.forces()
    one = want[:3]
    assert np.array_equal(want, np.tile(one, (40, 1))) and np.abs(one.sum(0)).max() < 1e-10
    for empty in ([], [none], [none, none]):
        b.reload(empty)
        if how == "run":
            b.run()
            b.sync()
        assert b.forces().shape == (0, 3)
        Es, Ea = b.energy()
        assert Ea.shape == (0, 1) and np.array_equal(Es, np.zeros((len(empty), 1)))
        b.reload(pairs)
        assert np.array_equal(b.forces(), want)
    b.close()
