"""Captured steps against steps launched one by one where a grid would otherwise take the resident loop on
both sides (DGFEM_RESIDENT=0): bit for bit, both integrators and precisions, with learned faces, runs that
the captured sequences do not divide, and successive runs of both integrators against the oracle."""
import numpy as np
import pytest

import dgfem_amd as dg
import test_gpu_api
import test_gpu_parity
import test_gpu_resident

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def launches_per_stage(monkeypatch):
    for name in ("DGFEM_KERNEL", "DGFEM_QUAD", "DGFEM_TET_MM", "DGFEM_POST_BRANCH"):
        monkeypatch.delenv(name, raising=False)
    monkeypatch.setenv("DGFEM_RESIDENT", "0")


@pytest.mark.parametrize("dim,order,n", [(2, 3, 12), (3, 2, 4), (3, 3, 3)])
@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
@pytest.mark.parametrize("integrator", [dg.DG_RK4, dg.DG_EULER])
@pytest.mark.parametrize("learned", [False, True])
def test_graph_equals_eager(dim, order, n, precision, integrator, learned, monkeypatch):
    print(f"case graph eager dim={dim} order={order} precision={precision} integrator={integrator} learned={learned}",
          flush=True)
    m = dg.box_mesh(dim, n, order, jitter=0.1, seed=n)
    bc = dg.resolve_bc_sides(m, [(0x3, 1), (0x3C if dim == 3 else 0xC, 2 if learned else 0)])
    net = None
    if learned:
        net = dg.to_bf16(dg.closure_init(order + 1 if dim == 2 else dg.num_nodes(2, order), seed=4, out_scale=0.1, dim=dim))
    create = dg.Solver.__init__
    out = []
    for use_graph in (True, False):
        def init(self, *args, **kw):
            create(self, *args, use_graph=use_graph, **kw)
            assert self.forms().resident == 0

        monkeypatch.setattr(dg.Solver, "__init__", init)
        out.append(test_gpu_resident._run(m, bc, order, 4, precision, "0", monkeypatch, integrator=integrator, net=net))
    for x, y in zip(*out):
        assert np.isfinite(x).any()
        np.testing.assert_array_equal(x, y)


def test_replay_of_the_parity_case():
    test_gpu_parity.test_graph_replay_equals_eager()


@pytest.mark.parametrize("use_graph", [True, False])
def test_successive_runs(use_graph):
    test_gpu_api.test_successive_runs_continue_the_state(use_graph)
