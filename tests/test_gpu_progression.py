"""Angular groups whose exponents form a progression x0 + k s (the reference's automatic scheme,
acsf.F90:276-363): one P^s per pair and lambda in place of a power per member.

The automatic scheme with fractional and integer steps, groups split at 16 members (whose second
part starts above xi = 1), one lambda only, a G4 progression and a ladder group beside one, over
rows of one entry up to periodic cells, against the FP64 oracle: values and energies 1e-10 and
forces 1e-9 of the largest value in FP64; in FP32 the features within 64 exponents' worth of FP32
rounding (xi eps = 16 x 6e-8 per term, so 1e-5) and the forces within the 1e-4 eV/A gate.
"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W

from test_gpu_workloads import F_RMSE_TOL, EV_BOHR_TO_EV_AA, _clusters, _oracle_all, ctx  # noqa: F401

pytestmark = pytest.mark.gpu
RC = 6.0 * fa.AA__BOHR


def _steps(ty, x0, s, n, lams, eta=0.005):
    lam = [l for _ in range(n) for l in lams]
    xi = [x0 + k * s for k in range(n) for _ in lams]
    return fa.GFunctions([ty] * len(xi), [RC] * len(xi), eta=W.eta_bohr([eta] * len(xi)), xi=xi,
                         lam=lam)


SETS = {
    "auto16": lambda: fa.GFunctions.auto(RC, 4, 16),             # step 15/7, 8 per lambda
    "auto12": lambda: fa.GFunctions.auto(RC, 4, 12),             # step 3
    "auto40": lambda: fa.GFunctions.auto(RC, 4, 40),             # groups of 16, 16 and 8 members
    "auto7_resolved": lambda: fa.GFunctions.auto(RC, 3, 7).species_resolved([1, 8]),
    "g4_one_lambda": lambda: fa.GFunctions.concat([fa.GFunctions.auto(RC, 3, 1),
                                                   _steps(4, 1.5, 0.75, 3, [-1.0])]),
    "beside_ladder": lambda: fa.GFunctions.concat(
        [fa.GFunctions.auto(RC, 3, 6), _steps(5, 1.0, 1.0, 2, [1.0, -1.0], 0.02)]),
}


@pytest.mark.parametrize("name", sorted(SETS))
@pytest.mark.parametrize("cells", ["clusters", "periodic"])
def test_progressions_match_oracle(ctx, name, cells):  # noqa: F811
    print("progression", name, cells, flush=True)
    geos = _clusters(5) if cells == "clusters" else [W.water_box(31, 22, 8.7), W.water_box(32, 7, 6.0)]
    g = SETS[name]()
    dims = [len(g), 8, 1]
    ns = fa.Netstat(g, [1, 8], dims, 0, W.random_params(dims, 2, 9))
    ctx.upload_model(ns)
    b = ctx.batch(geos, fa.FNET_FP64)
    ns = W.with_zscore(ns, b.acsf())
    b.close()
    ctx.upload_model(ns)
    G0, E0, F0 = _oracle_all(geos, ns)
    b = ctx.batch(geos, fa.FNET_FP64)
    assert np.abs(b.acsf() - G0).max() <= 1e-10 * max(1.0, np.abs(G0).max())
    assert np.abs(b.energy()[1] - E0).max() <= 1e-10 * max(1.0, np.abs(E0).max())
    assert np.abs(b.forces() - F0).max() <= 1e-9 * max(1.0, np.abs(F0).max())
    b.set_mode(fa.FNET_FP32)
    assert np.abs(b.acsf() - G0).max() <= 1e-5 * max(1.0, np.abs(G0).max())
    if cells == "periodic":
        rmse = np.sqrt(np.mean((b.forces() - F0) ** 2)) * EV_BOHR_TO_EV_AA
        assert rmse <= F_RMSE_TOL * max(1.0, np.abs(F0).max())
    b.close()
