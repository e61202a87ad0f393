"""Resident launches that are given up where blocks of learned faces take part: with no patience some
block, of elements or of learned faces, aborts the launch in one of its first exchanges. The whole run is
then done by launches per stage, bit for bit as without the resident loop."""
import numpy as np
import pytest

import dgfem_amd as dg
import test_gpu_resident

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,order,fields,n", [(2, 1, 4, 6), (2, 3, 5, 30), (2, 4, 4, 60), (3, 2, 4, 4), (3, 3, 5, 6)])
@pytest.mark.parametrize("integrator", [dg.DG_RK4, dg.DG_EULER])
def test_learned_faces_give_up(dim, order, fields, n, integrator, monkeypatch):
    print(f"case resident abort dim={dim} order={order} fields={fields} n={n} integrator={integrator}", flush=True)
    seen, close = [], dg.Solver.close

    def recording(self):
        if getattr(self, "_h", None):
            seen.append(self.forms())
        close(self)

    monkeypatch.setattr(dg.Solver, "close", recording)
    m = dg.box_mesh(dim, n, order, jitter=0.1, seed=n)
    bc = dg.resolve_bc_sides(m, [(0x3, dg.DG_BC_REFLECTING), (0x3C if dim == 3 else 0xC, dg.DG_BC_LEARNED)])
    net = dg.to_bf16(dg.closure_init(order + 1 if dim == 2 else dg.num_nodes(2, order), seed=4, out_scale=0.1, dim=dim))
    args = (m, bc, order, fields, dg.DG_MIXED)
    kw = dict(integrator=integrator, steps=60, save=50, net=net)
    a = test_gpu_resident._run(*args, "0", monkeypatch, **kw)
    b = test_gpu_resident._run(*args, "1", monkeypatch, patience="0", **kw)
    assert [f.resident_aborts for f in seen] == [0, 1]
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)
