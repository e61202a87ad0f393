"""The lane-per-field stage kernel (DGFEM_QUAD=1: at any size; by default from 163,840 order-3
tetrahedra in mixed precision) against the matrix-core volume variant (DGFEM_KERNEL=vm): element
counts of less than one, one and several groups of 16 with and without a remainder, every kind of
wall, both integrators, the right-hand side, sources, observers and save steps. The two differ in
FP32 rounding only; the bar is that of test_gpu_resident.py."""
import numpy as np
import pytest

import dgfem_amd as dg

pytestmark = pytest.mark.gpu

TOL = 3e-6
V0, RHO0, C0 = (30.0, -20.0, 10.0), 1.225, 340.0


def _solver(m, bc, env, monkeypatch, net):
    for name in ("DGFEM_KERNEL", "DGFEM_QUAD"):
        monkeypatch.delenv(name, raising=False)
    monkeypatch.setenv("DGFEM_RESIDENT", "0")
    monkeypatch.setenv(*env)
    s = dg.Solver(m.node_coords, m.element_vertices, 3, bc, v0=V0, rho0=RHO0, c0=C0, precision=dg.DG_MIXED,
                  steps_per_graph=5)
    if net is not None:
        s.set_closure(net)
    return s


@pytest.mark.parametrize("n", [1, 2, 3, 5])
@pytest.mark.parametrize("walls", ["absorbing", "reflecting", "learned", "all"])
@pytest.mark.parametrize("integrator", [dg.DG_RK4, dg.DG_EULER])
def test_quad_equals_vm(n, walls, integrator, monkeypatch):
    print(f"case quad n={n} walls={walls} integrator={integrator}", flush=True)
    m = dg.box_mesh(3, n, 3, jitter=0.1, seed=n)
    sides = {"absorbing": [(0x3F, 0)], "reflecting": [(0x3F, 1)], "learned": [(0x3F, 2)],
             "all": [(0x03, 0), (0x0C, 1), (0x30, 2)]}[walls]
    bc = dg.resolve_bc_sides(m, sides)
    net = dg.to_bf16(dg.closure_init(10, seed=4, out_scale=0.1, dim=3)) if walls in ("learned", "all") else None
    X = m.node_coords.reshape(-1, 3)
    rng = np.random.default_rng(n)
    u = rng.normal(0, 0.1, (4, len(X))) * np.array([[1.0], [2e-3], [2e-3], [2e-3]])
    u[0] += np.exp(-((X - 0.2) ** 2).sum(1) / 0.3)
    out = []
    for env in (("DGFEM_KERNEL", "vm"), ("DGFEM_QUAD", "1")):
        s = _solver(m, bc, env, monkeypatch, net)
        dt = s.info().min_inradius / (500.0 * 7) * (0.1 if integrator == dg.DG_EULER else 1.0)
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
            assert np.linalg.norm(a - b) <= f * TOL * np.linalg.norm(a), np.linalg.norm(a - b) / np.linalg.norm(a)
