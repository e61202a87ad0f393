"""A batch whose resident launches end before its steps do (DGFEM_RESIDENT_LAUNCHES: the launch after that
many, of 256 steps each, is refused): launches per stage go on at the step reached. State, residuals and
observers of the whole batch against a launch per stage from its start, with a source active across the
boundary; and the step of a non-finite state before and after it."""
import numpy as np
import pytest

import dgfem_amd as dg
import test_gpu_resident

pytestmark = pytest.mark.gpu


@pytest.fixture
def forms(monkeypatch):
    seen, close = [], dg.Solver.close

    def recording(self):
        if getattr(self, "_h", None):
            seen.append(self.forms())
        close(self)

    monkeypatch.setattr(dg.Solver, "close", recording)
    return seen


@pytest.mark.parametrize("launches", [0, 1, 2])
@pytest.mark.parametrize("integrator", [dg.DG_RK4, dg.DG_EULER])
@pytest.mark.parametrize("precision,learned", [(dg.DG_FP64, False), (dg.DG_MIXED, False), (dg.DG_MIXED, True)])
def test_resume(launches, integrator, precision, learned, forms, monkeypatch):
    print(f"case resume launches={launches} integrator={integrator} precision={precision} learned={learned}", flush=True)
    m = dg.box_mesh(2, 20, 2, jitter=0.1, seed=1)
    bc = dg.resolve_bc_sides(m, [(0x3, dg.DG_BC_REFLECTING), (0xC, dg.DG_BC_LEARNED if learned else dg.DG_BC_ABSORBING)])
    net = dg.to_bf16(dg.closure_init(3, seed=4, out_scale=0.1, dim=2)) if learned else None
    # 512 steps and a rest that the library's 8-step graphs do not divide
    args, kw = (m, bc, 2, 4, precision), dict(integrator=integrator, steps=531, save=532, net=net)
    want = test_gpu_resident._run(*args, "0", monkeypatch, **kw)
    monkeypatch.setenv("DGFEM_RESIDENT_LAUNCHES", str(launches))
    got = test_gpu_resident._run(*args, "1", monkeypatch, **kw)
    assert (forms[1].resident_launches, forms[1].resident_aborts, forms[1].resident) == (launches, 1, 0)
    if launches == 0:
        for x, y in zip(got, want):
            np.testing.assert_array_equal(x, y)
    # the bar of test_gpu_resident.py is for 50 steps; rounding adds up at random (forward Euler: a tenth of the step)
    tol = test_gpu_resident.TOL[dg.DG_MIXED if learned else precision]
    test_gpu_resident._close(got, want, tol * (np.sqrt(531 / 50) if integrator == dg.DG_RK4 else 1.0))


@pytest.mark.parametrize("residuals", [True, False])
@pytest.mark.parametrize("bad", [100, 300, 520])
@pytest.mark.parametrize("launches", [1, 2])
def test_non_finite_step(launches, bad, residuals, forms, monkeypatch):
    """A source that turns infinite: the same step is reported whichever way it was done."""
    print(f"case resume non-finite launches={launches} bad={bad} residuals={residuals}", flush=True)
    m = dg.box_mesh(2, 12, 3, jitter=0.1, seed=2)
    at = []
    for resident in "01":
        monkeypatch.setenv("DGFEM_RESIDENT", resident)
        monkeypatch.setenv("DGFEM_RESIDENT_LAUNCHES", str(launches))
        s = dg.Solver(m.node_coords, m.element_vertices, 3, None, rho0=1.225, c0=340.0, precision=dg.DG_MIXED)
        dt = s.info().min_inradius / (340.0 * 7 * 2)
        assert s.add_table_source(0.0, 0.0, 0.0, 0.3, lambda t: np.inf if t > (bad - 0.5) * dt else np.sin(900 * t)) > 0
        s.set_state(np.zeros(s.state_shape))
        with pytest.raises(dg.DGError) as e:
            s.run(0.0, 599.5 * dt, dt, 1e9, residuals=residuals)
        assert e.value.code == dg.DG_ERR_NONFINITE
        at.append(e.value.result.steps)
        s.close()
    assert forms[1].resident_launches == launches and forms[1].resident_aborts == 1
    assert at[0] == at[1] and abs(at[0] - bad) <= 1
