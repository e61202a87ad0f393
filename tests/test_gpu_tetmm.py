"""The matrix-core stage kernel of tetrahedra (DGFEM_TET_MM=1: at any size; FP64 of order 4 and 5, mixed
precision of order 4) against the thread-per-node kernel (DGFEM_KERNEL=valu): element counts of less
than one, one and several groups of 16 with and without a remainder, every kind of wall, both
integrators, 4 and 5 fields, the right-hand side, sources, observers and save steps. The two differ
in the order of sums of at most 252 terms, some of which cancel: the bar is 500 units of 2.2e-16 in
FP64 and 50 units of 6.0e-8 (3e-6, the bar between the other kernels of that precision) in mixed
precision for fields, four times that for the residuals, which are sums of squared differences of
states."""
import numpy as np
import pytest

import dgfem_amd as dg

pytestmark = pytest.mark.gpu

TOL = {dg.DG_FP64: 1.1e-13, dg.DG_MIXED: 3e-6}
V0, RHO0, C0 = (30.0, -20.0, 10.0), 1.225, 340.0


@pytest.mark.parametrize("walls", ["absorbing", "reflecting", "both"])
@pytest.mark.parametrize("fields", [4, 5])
@pytest.mark.parametrize("precision,order,n", [(dg.DG_FP64, p, n) for p in (4, 5) for n in (1, 2, 3)] +
                         [(dg.DG_MIXED, 4, n) for n in (1, 2, 3)])
@pytest.mark.parametrize("integrator", [dg.DG_RK4, dg.DG_EULER])
def test_matrix_core_equals_valu(order, n, walls, fields, precision, integrator, monkeypatch):
    print(f"case tetmm p={order} n={n} walls={walls} fields={fields} precision={precision} integrator={integrator}", flush=True)
    m = dg.box_mesh(3, n, order, jitter=0.1, seed=n)
    bc = dg.resolve_bc_sides(m, {"absorbing": [(0x3F, 0)], "reflecting": [(0x3F, 1)],
                                 "both": [(0x0F, 0), (0x30, 1)]}[walls])
    X = m.node_coords.reshape(-1, 3)
    rng = np.random.default_rng(n)
    u = rng.normal(0, 0.1, (fields, len(X))) * np.array([1.0, 2e-3, 2e-3, 2e-3, 1e-5][:fields])[:, None]
    u[0] += np.exp(-((X - 0.2) ** 2).sum(1) / 0.3)
    out = []
    monkeypatch.setenv("DGFEM_RESIDENT", "0")
    for kernel in ("valu", None):
        monkeypatch.delenv("DGFEM_KERNEL", raising=False)
        monkeypatch.setenv("DGFEM_TET_MM", "1")
        if kernel:
            monkeypatch.setenv("DGFEM_KERNEL", kernel)
        s = dg.Solver(m.node_coords, m.element_vertices, order, bc, v0=V0, rho0=RHO0, c0=C0,
                      fields=dg.DG_FIELDS_LEE5 if fields == 5 else dg.DG_FIELDS_REF4, precision=precision,
                      steps_per_graph=5)
        dt = s.info().min_inradius / (500.0 * (2 * order + 1)) * (0.1 if integrator == dg.DG_EULER else 1.0)
        k = s.rhs(u, dt)
        s.add_monopole(0.1, -0.1, 0.0, 1.2 / n, 0.3, 900.0, 0.2, 1.0)
        s.add_observer(0.5, 0.4, 0.3, 1.2 / n)
        s.set_state(u)
        r = s.run(0.0, 29.5 * dt, dt, 10.5 * dt, integrator=integrator)
        assert r.steps == 30
        out.append((k, s.get_state(), r.residuals, r.observers))
        s.close()
    for x, y, f, axis in zip(*out, (1.0, 1.0, 4.0, 1.0), (0, 0, 1, 2)):
        assert np.linalg.norm(x) > 0
        for a, b in zip(np.moveaxis(x, axis, 0), np.moveaxis(y, axis, 0)):  # every field by itself, records as series
            assert np.linalg.norm(a - b) <= f * TOL[precision] * np.linalg.norm(a), np.linalg.norm(a - b) / np.linalg.norm(a)
