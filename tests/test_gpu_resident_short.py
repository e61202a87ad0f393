"""Short batches (calls of few steps, saves every few steps) of a grid that has the resident loop: launched
per stage, kernel by kernel at first and captured later; the loop still takes the longer ones."""
import numpy as np
import pytest

import dgfem_amd as dg
import test_gpu_resident

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("integrator", [dg.DG_RK4, dg.DG_EULER])
@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
def test_short_batches(precision, integrator, use_graph, monkeypatch):
    print(f"case resident short precision={precision} integrator={integrator} graph={use_graph}", flush=True)
    for name in ("DGFEM_KERNEL", "DGFEM_POST_BRANCH", "DGFEM_RESIDENT_LAUNCHES", "DGFEM_RESIDENT_PATIENCE"):
        monkeypatch.delenv(name, raising=False)
    m = dg.box_mesh(2, 12, 3, jitter=0.1, seed=2)
    X = m.node_coords.reshape(-1, 3)
    u = np.zeros((4, len(X)))
    u[0] = np.exp(-(X ** 2).sum(1) / 0.1)
    out, counts = [], []
    for resident in "01":
        monkeypatch.setenv("DGFEM_RESIDENT", resident)
        s = dg.Solver(m.node_coords, m.element_vertices, 3, None, rho0=1.225, c0=340.0, precision=precision,
                      use_graph=use_graph, steps_per_graph=4)
        dt = s.info().min_inradius / (340.0 * 7 * 8) * (0.1 if integrator == dg.DG_EULER else 1.0)
        s.add_monopole(0.1, -0.1, 0.0, 0.3, 0.2, 900.0, 0.2, 1.0)
        s.add_observer(0.4, 0.3, 0.0, 0.3)
        s.set_state(u)
        t, rec, seen = 0.0, [], []

        def run(steps, h, save=1e9):
            nonlocal t
            r = s.run(t, t + (steps - 0.5) * h, h, save, integrator=integrator)
            assert r.steps == steps
            t += steps * h
            rec.append((r.residuals, r.observers))
            seen.append(s.forms().resident_launches)

        for _ in range(20):
            run(1, dt)
        run(6, dt)
        for _ in range(3):
            run(5, dt)
        run(40, dt)
        run(12, dt, save=2.5 * dt)  # saves at step 0 and then every 3: batches of 3
        for _ in range(2):
            run(2, 0.5 * dt)
        out.append((s.get_state(), *(np.concatenate(x) for x in zip(*rec))))
        counts.append(seen)
        s.close()
    assert counts[0] == [0] * 28
    assert counts[1] == [0] * 20 + [1] * 4 + [2] * 4
    # 107 steps of at most an eighth of the bar's
    test_gpu_resident._close(*out[::-1], test_gpu_resident.TOL[precision])


@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
@pytest.mark.parametrize("steps", [1, 5, 6])
def test_same_call_same_bits(precision, steps, monkeypatch):
    """A call from the same state gives the same bits each time: the first, which captures nothing, those
    after the graphs are captured, with and without the resident loop's calls of another length between."""
    print(f"case resident same call precision={precision} steps={steps}", flush=True)
    monkeypatch.delenv("DGFEM_RESIDENT", raising=False)
    m = dg.box_mesh(2, 12, 3, jitter=0.1, seed=2)
    X = m.node_coords.reshape(-1, 3)
    u = np.zeros((4, len(X)))
    u[0] = np.exp(-(X ** 2).sum(1) / 0.1)
    s = dg.Solver(m.node_coords, m.element_vertices, 3, None, rho0=1.225, c0=340.0, precision=precision)
    dt = s.info().min_inradius / (340.0 * 7)
    s.add_observer(0.4, 0.3, 0.0, 0.3)
    first = None
    for k in range(24):
        if k % 5 == 4:
            s.run_steps(20, dt)
        s.set_state(u)
        r = s.run_steps(steps, dt)
        got = s.get_state(), r.residuals, r.observers
        if first is None:
            first = got
        for x, y in zip(got, first):
            np.testing.assert_array_equal(x, y)
    s.close()
