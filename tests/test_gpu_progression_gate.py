"""FP32 and BF16 forces of progression groups against the 1e-4 eV/A gate itself, with networks scaled so
that the largest force is 2 eV/A, as in a perturbed crystal or liquid: clusters and periodic cells."""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_progression import SETS
from test_gpu_workloads import F_RMSE_TOL, EV_BOHR_TO_EV_AA, _clusters, _oracle_all, ctx  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", sorted(SETS))
@pytest.mark.parametrize("cells", ["clusters", "periodic"])
def test_force_gate(ctx, name, cells):  # noqa: F811
    geos = _clusters(5) if cells == "clusters" else [W.water_box(31, 22, 8.7), W.water_box(32, 7, 6.0)]
    g = SETS[name]()
    dims = [len(g), 8, 1]
    ns = fa.Netstat(g, [1, 8], dims, 0, W.random_params(dims, 2, 9))
    ctx.upload_model(ns)
    b = ctx.batch(geos, fa.FNET_FP64)
    ns = W.with_zscore(ns, b.acsf())
    ns.params[:, 8 * len(g):8 * len(g) + 8] *= 2.0 / (np.abs(_oracle_all(geos, ns)[2]).max() * EV_BOHR_TO_EV_AA)
    F0 = _oracle_all(geos, ns)[2]
    assert abs(np.abs(F0).max() * EV_BOHR_TO_EV_AA - 2.0) < 1e-9
    ctx.upload_model(ns)
    for mode in (fa.FNET_FP32, fa.FNET_BF16):
        b.set_mode(mode)
        rmse = np.sqrt(np.mean((b.forces() - F0) ** 2)) * EV_BOHR_TO_EV_AA
        print(name, cells, mode, "RMSE eV/A", rmse, flush=True)
        assert rmse <= F_RMSE_TOL
    b.close()
