"""Learned faces with an infinite weight in a hidden layer: the unit saturates (tanh = +-1) and the exterior
state is finite, in mixed precision as in FP64 (whose kernel sums each unit in one FP32 chain), with a
launch per stage and in the resident loop."""
import numpy as np
import pytest

import dgfem_amd as dg
from cases import rel_l2, smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,order", [(2, 3), (3, 2)])
@pytest.mark.parametrize("layer", [1, 2])
@pytest.mark.parametrize("bits", [0x7f80, 0xff80, 0x7f7f])
def test_infinite_hidden_weight(dim, order, layer, bits, monkeypatch):
    print(f"case closure weights dim={dim} layer={layer} bits={bits:#x}", flush=True)
    m = dg.box_mesh(dim, 4 if dim == 2 else 2, order, jitter=0.1, seed=1)
    nfp = order + 1 if dim == 2 else dg.num_nodes(2, order)
    nin = dim * nfp + 2
    net = dg.to_bf16(dg.closure_init(nfp, seed=4, out_scale=0.1, dim=dim))
    net[{1: 5 * nin + 1, 2: 64 * nin + 64 + 7 * 64 + 5}[layer]] = bits
    u = smooth_state(m)
    out = []
    for precision, resident in ((dg.DG_FP64, "0"), (dg.DG_MIXED, "0"), (dg.DG_MIXED, "1")):
        monkeypatch.setenv("DGFEM_RESIDENT", resident)
        s = dg.Solver(m.node_coords, m.element_vertices, order, np.full(m.face_side.shape, dg.DG_BC_LEARNED, np.int8),
                      v0=(30.0, -20.0, 10.0 * (dim - 2)), rho0=1.225, c0=100.0, precision=precision)
        s.set_closure(net)
        k = s.rhs(u, 1e-5)
        s.set_state(u)
        s.run_steps(4, 1e-7)
        out.append((k, s.get_state()))
        s.close()
    for k, state in out[1:]:
        for f in range(dim + 1):
            assert np.isfinite(out[0][0][f]).all()
            assert rel_l2(k[f], out[0][0][f]) < 2e-5 and rel_l2(state[f], out[0][1][f]) < 2e-6
