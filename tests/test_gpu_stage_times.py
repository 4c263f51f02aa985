"""Device times of a step: each stage takes some time and they add up to the step, for batches searched
directly, with cell lists and with both, with results in pinned memory and without, in steady state and
through the host.  (The host's clock and the device's are not compared: they differ by per cents.)"""
import numpy as np
import pytest

import fortnet_amd as fa
from fortnet_amd import workloads as W
from test_gpu_neighbours import ctx  # noqa: F401

pytestmark = pytest.mark.gpu
RC = 4.0 * fa.AA__BOHR
KINDS = {"direct": [3], "bins": [6], "bins_then_direct": [6, 3], "direct_then_bins": [3, 6],
         "large": [14, 3]}


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_stage_times(ctx, kind, graph):  # noqa: F811
    print(kind, graph, flush=True)
    dims = [4, 8, 1]
    g = fa.GFunctions([2, 2, 5, 5], [RC] * 4, eta=[0.1, 0.02, 0.01, 0.01], xi=[0, 0, 1, 4],
                      lam=[0, 0, 1.0, -1.0])
    ctx.upload_model(fa.Netstat(g, [14], dims, 0, W.random_params(dims, 1, 5)))
    b = ctx.batch([W.si_diamond(n, n, n, 0.1, n) for n in KINDS[kind]], fa.FNET_FP32)
    ctx.set_graph(graph)
    for step in range(4):  # the first step goes through the host
        b.run()
        b.sync()
        whole, stages = ctx.step_time(), b.stage_times()
        print(step, b.graph_replayed(), whole, stages, flush=True)
        assert whole > 0.0
        if b.graph_replayed():
            assert stages[0] == whole
        else:
            assert (stages > 0.0).all() and abs(stages.sum() - whole) <= 1e-3 * whole
    ctx.set_graph(False)
    b.close()
