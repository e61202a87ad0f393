"""Runs of both integrators after one another on one context of the lane-per-field stage kernel, on a
mesh of more than 32,768 elements, where its forward-Euler grid has more blocks than that of the last
RK4 stage: every run's residuals and state are those of a fresh context set to the same state, bit for
bit, also after a forward-Euler run that ended in non-finite values."""
import numpy as np
import pytest

import dgfem_amd as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
def test_residuals_after_the_other_integrator(use_graph, monkeypatch):
    print(f"case quad integrators graph={use_graph}", flush=True)
    monkeypatch.delenv("DGFEM_KERNEL", raising=False)
    monkeypatch.setenv("DGFEM_QUAD", "1")
    m = dg.box_mesh(3, 18, 3, jitter=0.1, seed=3)
    assert m.K > 32768
    X = m.node_coords.reshape(-1, 3)
    u = np.zeros((4, len(X)))
    u[0] = np.exp(-((X - 0.2) ** 2).sum(1) / 0.3)

    def solver():
        return dg.Solver(m.node_coords, m.element_vertices, 3, None, v0=(30.0, -20.0, 10.0), rho0=1.225, c0=340.0,
                         precision=dg.DG_MIXED, use_graph=use_graph, steps_per_graph=3)

    def run(s, integrator):
        dt = s.info().min_inradius / (500.0 * 7) * (0.1 if integrator == dg.DG_EULER else 1.0)
        s.set_state(u)
        r = s.run_steps(5, dt, integrator=integrator)
        return r.residuals, s.get_state()

    fresh = {}
    for integrator in (dg.DG_RK4, dg.DG_EULER):
        s = solver()
        fresh[integrator] = run(s, integrator)
        s.close()
    s = solver()
    for integrator in (dg.DG_EULER, dg.DG_RK4, dg.DG_EULER, dg.DG_RK4):
        for got, want in zip(run(s, integrator), fresh[integrator]):
            np.testing.assert_array_equal(got, want)
    s.set_state(np.full_like(u, np.inf))
    with pytest.raises(dg.DGError) as e:
        s.run_steps(3, 1e-6, integrator=dg.DG_EULER)
    assert e.value.code == dg.DG_ERR_NONFINITE
    for got, want in zip(run(s, dg.DG_RK4), fresh[dg.DG_RK4]):
        np.testing.assert_array_equal(got, want)
    s.close()
