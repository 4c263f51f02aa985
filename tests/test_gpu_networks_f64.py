"""FP64 networks on the matrix cores (16 atoms per block, outputs in blocks of 16, K in steps of 4)
against the FP64 oracle: layer widths around the block edges, one to eight outputs, two to five
layers, one to several hundred atoms of one or three elements, and a network too wide for a
block's LDS (which keeps the scalar kernels).  Outputs and weight gradients must agree to 1e-11 of
the largest value: sums of up to 256 products in another order differ by 256 eps = 6e-14, times the
amplification of a few layers.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [  # hidden and output widths, activations, atoms
    ([1], 9, 1), ([3], 0, 15), ([1, 1], 0, 16), ([15, 8], 1, 17), ([16, 1], 4, 40),
    ([17, 33, 1], 0, 300), ([20, 20, 20, 2], 7, 65), ([32, 128, 1], 6, 33), ([100, 100, 3], 0, 130),
    ([240, 250, 1], 0, 20), ([31, 5], 5, 700),
]


@pytest.fixture(scope="module")
def ctx():
    c = fa.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("widths,act,atoms", SHAPES)
def test_fp64_networks_match_oracle(ctx, widths, act, atoms):
    print("networks", widths, act, atoms, flush=True)
    rng = np.random.default_rng(atoms)
    rc = 4.0
    nsp = 1 if atoms < 100 else 3
    z = np.array([6, 8, 14])[:nsp]
    g = fa.GFunctions([2] * 5, [rc] * 5, eta=[0.1, 0.3, 0.5, 0.9, 1.5])
    dims = [5] + list(widths)
    nout = dims[-1]
    params = W.random_params(dims, nsp, 3)
    params += 0.1 * rng.standard_normal(params.shape)  # biases too
    L = 1.7 * max(atoms, 8) ** (1.0 / 3.0)
    sp = rng.integers(0, nsp, atoms)
    geo = fa.Geometry(rng.uniform(0, L, (atoms, 3)), z[sp], sp)
    ns = fa.Netstat(g, z, dims, act, params, np.full(5, 0.3), np.full(5, 1.5), n_global=0)
    ctx.upload_model(ns)
    b = ctx.batch([geo], fa.FNET_FP64)
    gf = O.GFunctions(g.type, g.rcut, g.eta, g.rs, g.kappa, g.lam, g.xi, g.atomid, g.z1, g.z2)
    st = O.Structure(geo.coords, geo.latvecs, 0, geo.atnum)
    X = O.zscore(O.acsf(st, gf), ns.zmean, ns.zstd)
    nets = O.Nets(dims, ns.activation, params)
    E0 = nets.predict(X, geo.species)
    close = lambda a, c: np.abs(a - c).max() <= 1e-11 * max(1.0, np.abs(c).max())
    assert close(b.energy()[1], E0)
    J = nets.jacobian(X, geo.species)
    F = b.forces()
    for t in range(nout):
        F0 = O.acsf_adjoint(st, gf, J[:, t, :] * O.zscale(ns.zstd, gf.n)[None, :])
        assert close(F[:, 3 * t:3 * t + 3], F0.reshape(atoms, 3))
    at = rng.standard_normal((atoms, nout))
    grad, pred = b.train_gradients(None, at)
    g0 = np.zeros_like(params)
    nets.sys_train(X, geo.species, 0, None, at, np.ones(atoms), 1.0, g0)
    assert close(pred, E0)
    assert close(grad, g0)
    b.close()
