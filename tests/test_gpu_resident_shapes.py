"""The resident loop on the largest grids of each of its block shapes (more blocks per CU, several face
nodes per thread, operators in LDS) against a launch per stage: 4 and 5 fields, both precisions, walls
and learned faces; sources, observers, save steps and bars as in test_gpu_resident.py."""
import pytest

import dgfem_amd as dg
import test_gpu_resident

pytestmark = pytest.mark.gpu

# cells per side of the largest grids: (dim, order) -> {shape: n}; with 5 fields some shapes are passed over
WALLS = {dg.DG_FP64: {(2, 1): {1: 125}, (2, 2): {1: 118, 2: 125}, (2, 3): {1: 102}, (2, 4): {1: 92}, (2, 5): {1: 77},
                      (3, 1): {1: 13}, (3, 2): {1: 10}, (3, 3): {1: 9, 2: 11}},
         dg.DG_MIXED: {(2, 1): {1: 145, 2: 207}, (2, 2): {1: 118, 2: 145, 3: 162}, (2, 3): {1: 102, 2: 112, 3: 125},
                       (2, 4): {1: 92, 3: 103}, (2, 5): {1: 77, 3: 86}, (3, 1): {1: 15}, (3, 2): {1: 11},
                       (3, 3): {1: 10, 2: 12, 3: 13}}}
LEARNED = {dg.DG_MIXED: {(2, 1): {1: 143, 2: 202, 3: 226}, (2, 2): {1: 116, 2: 143, 3: 160},
                         (2, 3): {1: 101, 2: 110, 3: 123}, (2, 4): {1: 91, 3: 102}, (2, 5): {1: 76, 3: 85},
                         (3, 1): {1: 14}, (3, 2): {1: 11}, (3, 3): {1: 9, 2: 12, 3: 13}}}
# (precision, dim, order, fields, shape) whose blocks one of the earlier shapes already holds, or that is not built
SKIP = {(dg.DG_FP64, 3, 1, 5, 1), (dg.DG_FP64, 3, 2, 4, 1), (dg.DG_FP64, 3, 3, 4, 1), (dg.DG_MIXED, 2, 1, 4, 1),
        (dg.DG_MIXED, 3, 3, 4, 1)}
CASES = [(precision, dim, order, fields, shape, n, learned)
         for learned, table in ((False, WALLS), (True, LEARNED)) for precision, rows in table.items()
         for (dim, order), shapes in rows.items() for shape, n in shapes.items() for fields in (4, 5)
         if (precision, dim, order, fields, shape) not in SKIP]


@pytest.mark.parametrize("precision,dim,order,fields,shape,n,learned", CASES)
def test_largest_grids(precision, dim, order, fields, shape, n, learned, monkeypatch):
    print(f"case shapes precision={precision} dim={dim} order={order} fields={fields} shape={shape} n={n} learned={learned}",
          flush=True)
    seen, close = [], dg.Solver.close

    def recording(self):
        if getattr(self, "_h", None):
            seen.append(self.forms())
        close(self)

    monkeypatch.setattr(dg.Solver, "close", recording)
    m = dg.box_mesh(dim, n, order, jitter=0.1, seed=n)
    bc = dg.resolve_bc_sides(m, [(0x3, 1), (0x3C if dim == 3 else 0xC, 2 if learned else 0)])
    net = None
    if learned:
        net = dg.to_bf16(dg.closure_init(order + 1 if dim == 2 else dg.num_nodes(2, order), seed=4, out_scale=0.1, dim=dim))
    args, kw = (m, bc, order, fields, precision), dict(steps=20, save=8, net=net)
    a = test_gpu_resident._run(*args, "1", monkeypatch, **kw)
    b = test_gpu_resident._run(*args, "0", monkeypatch, **kw)
    # batches of 8, 8 and 4 steps: the last is launched per stage
    assert (seen[0].resident_shape, seen[0].resident, seen[0].resident_launches, seen[0].resident_aborts) == (shape, 1, 2, 0)
    assert seen[1].resident_launches == 0
    test_gpu_resident._close(a, b, test_gpu_resident.TOL[precision])
