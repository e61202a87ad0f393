"""The resident time loop of small grids (one launch for many steps, exchanges between blocks) against
a launch per stage (DGFEM_RESIDENT=0) on the same case: every (dim, order, fields) it is built for and
both precisions, from a grid of one block over a partial last block to the shapes of larger grids;
overlapping sources, one of them switching off, a table source, observers on and off source nodes,
save steps, both integrators, runs longer than one launch; the step of a non-finite state; and the
way back to launches per stage when a block would have to wait."""
import threading

import numpy as np
import pytest

import dgfem_amd as dg

pytestmark = pytest.mark.gpu

RHO0, C0 = 1.225, 340.0
# The two paths differ in rounding only. One right-hand side of FP32 operands is 1e-7..4.4e-7 off its
# FP64 value; a stage adds at most a fifth of it to the state, 4 x 50 stages at random: 0.2 * 4.4e-7 *
# sqrt(200) = 1.2e-6, twice for the two paths. FP64: 2^-29 of that.
TOL = {dg.DG_MIXED: 3e-6, dg.DG_FP64: 6e-15 * 2}


def _run(m, bc, order, fields, precision, resident, monkeypatch, integrator=dg.DG_RK4, steps=50, save=17, patience=None,
         net=None):
    monkeypatch.setenv("DGFEM_RESIDENT", resident)
    if patience is not None:
        monkeypatch.setenv("DGFEM_RESIDENT_PATIENCE", patience)
    dim = m.dim
    s = dg.Solver(m.node_coords, m.element_vertices, order, bc, v0=(30.0, -20.0, 10.0 if dim == 3 else 0.0), rho0=RHO0,
                  c0=C0, fields=dg.DG_FIELDS_LEE5 if fields == 5 else dg.DG_FIELDS_REF4, precision=precision,
                  steps_per_graph=8)
    if net is not None:
        s.set_closure(net)
    X = m.node_coords.reshape(-1, 3)
    u = np.zeros(s.state_shape)
    u[0] = np.exp(-((X - 0.2 * np.array([1, 1, dim - 2])) ** 2).sum(1) / 0.1)
    u[1] = 1e-3 * np.sin(3 * X[:, 1])
    if fields == 5:
        u[4] = u[0] / C0 ** 2
    h = 2.0 / m.n
    dt = s.info().min_inradius / (500.0 * (2 * order + 1)) * (0.1 if integrator == dg.DG_EULER else 1.0)
    s.add_monopole(0.1, -0.1, 0.0, 1.1 * h, 0.3, 900.0, 0.2, 20 * dt)
    s.add_monopole(0.0, 0.0, 0.0, 1.1 * h, 0.2, 700.0, 0.0, 1.0)
    s.add_table_source(-0.5, -0.5, 0.0, 1.1 * h, lambda t: 0.1 * np.cos(3000.0 * t) if t < 30 * dt else None)
    s.add_observer(0.6, 0.5, 0.0, 1.1 * h)
    s.add_observer(0.1, -0.1, 0.0, 1.1 * h)
    s.add_observer(5.0, 5.0, 5.0, 0.1)  # no node: NaN records
    s.set_state(u)
    r = s.run(0.0, (steps - 0.5) * dt, dt, (save - 0.5) * dt, integrator=integrator)
    assert r.steps == steps and len(r.saves) >= steps // save
    out = s.get_state(), r.residuals, r.observers
    s.close()
    return out


def _close(a, b, tol):
    for x, y, f in zip(a, b, (1.0, 4.0, 1.0)):  # a residual is the square of a difference of states
        assert np.array_equal(np.isnan(x), np.isnan(y))
        x, y = np.nan_to_num(x), np.nan_to_num(y)
        assert np.linalg.norm(x - y) <= f * tol * np.linalg.norm(y), np.linalg.norm(x - y) / np.linalg.norm(y)


CASES = [(2, p, nf, n) for p, nf, n in ((1, 4, 2), (1, 5, 40), (1, 4, 120), (2, 4, 9), (2, 5, 70), (2, 4, 110), (3, 4, 3),
                                        (3, 5, 30), (3, 4, 90), (4, 4, 5), (4, 5, 50), (4, 4, 80), (5, 4, 4), (5, 5, 40),
                                        (5, 4, 60))]
CASES += [(3, p, nf, n) for p, nf, n in ((1, 4, 2), (1, 5, 9), (1, 4, 13), (2, 4, 3), (2, 5, 9), (2, 4, 11), (3, 4, 2),
                                         (3, 5, 7), (3, 4, 11))]


@pytest.mark.parametrize("dim,order,fields,n", CASES)
@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
def test_resident_equals_launch_per_stage(dim, order, fields, n, precision, monkeypatch):
    print(f"case resident dim={dim} order={order} fields={fields} n={n} precision={precision}", flush=True)
    m = dg.box_mesh(dim, n, order, jitter=0.1, seed=n)
    bc = dg.resolve_bc_sides(m, [(0x3, dg.DG_BC_REFLECTING), (0x3C if dim == 3 else 0xC, dg.DG_BC_ABSORBING)])
    args = (m, bc, order, fields, precision)
    _close(_run(*args, "1", monkeypatch), _run(*args, "0", monkeypatch), TOL[precision])


@pytest.mark.parametrize("dim,order,fields,n", [(2, 1, 5, 2), (2, 1, 4, 100), (2, 2, 4, 90), (2, 3, 5, 9), (2, 3, 4, 95),
                                                (2, 4, 4, 100), (2, 5, 4, 40), (3, 1, 4, 9), (3, 2, 5, 3), (3, 3, 4, 2),
                                                (3, 3, 4, 11)])
@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
def test_resident_learned_faces(dim, order, fields, n, precision, monkeypatch):
    """Learned faces on all but one pair of sides, evaluated by blocks of their own; the network is
    FP32 in both precisions."""
    print(f"case resident learned dim={dim} order={order} fields={fields} n={n} precision={precision}", flush=True)
    m = dg.box_mesh(dim, n, order, jitter=0.1, seed=n)
    bc = dg.resolve_bc_sides(m, [(0x3, dg.DG_BC_REFLECTING), (0x3C if dim == 3 else 0xC, dg.DG_BC_LEARNED)])
    nfp = order + 1 if dim == 2 else dg.num_nodes(2, order)
    net = dg.to_bf16(dg.closure_init(nfp, seed=4, out_scale=0.1, dim=dim))
    args = (m, bc, order, fields, precision)
    _close(_run(*args, "1", monkeypatch, net=net), _run(*args, "0", monkeypatch, net=net), TOL[dg.DG_MIXED])


@pytest.mark.parametrize("dim,order,n", [(2, 2, 20), (3, 2, 5)])
@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
def test_resident_euler_and_long_runs(dim, order, n, precision, monkeypatch):
    print(f"case resident euler dim={dim} precision={precision}", flush=True)
    m = dg.box_mesh(dim, n, order, jitter=0.1, seed=1)
    args = (m, None, order, 4, precision)
    # 600 steps without a save: three launches; 600 stages of a tenth the step
    kw = dict(integrator=dg.DG_EULER, steps=600, save=601)
    _close(_run(*args, "1", monkeypatch, **kw), _run(*args, "0", monkeypatch, **kw), TOL[precision])


@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
def test_waiting_block_falls_back(precision, monkeypatch):
    """With no patience a block that finds a mailbox empty aborts the launch: the batch is then done by
    launches per stage, bit for bit as without the resident loop."""
    print(f"case resident fallback precision={precision}", flush=True)
    m = dg.box_mesh(2, 40, 3, jitter=0.1, seed=3)
    args = (m, None, 3, 4, precision)
    a = _run(*args, "0", monkeypatch, steps=300, save=290)
    b = _run(*args, "1", monkeypatch, steps=300, save=290, patience="0")
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("residuals", [True, False])
def test_non_finite_step(residuals, monkeypatch):
    """An unstable step: both paths report the first step that left a non-finite value."""
    print(f"case resident non-finite residuals={residuals}", flush=True)
    m = dg.box_mesh(2, 12, 3, jitter=0.1, seed=2)
    X = m.node_coords.reshape(-1, 3)
    u = np.zeros((4, len(X)))
    u[0] = np.exp(-(X ** 2).sum(1) / 0.1)
    at = []
    for resident in ("0", "1"):
        monkeypatch.setenv("DGFEM_RESIDENT", resident)
        s = dg.Solver(m.node_coords, m.element_vertices, 3, None, rho0=RHO0, c0=C0, precision=dg.DG_MIXED)
        s.set_state(u)
        dt = 40 * s.info().min_inradius / (C0 * 7)
        with pytest.raises(dg.DGError) as e:
            s.run(0.0, 399.5 * dt, dt, 1e9, residuals=residuals)
        assert e.value.code == dg.DG_ERR_NONFINITE
        at.append(e.value.result.steps)
        s.close()
    assert at[0] == at[1] > 1


def test_two_threads(monkeypatch):
    """Two solvers stepping at the same time from two host threads, each as if it were alone."""
    print("case resident two threads", flush=True)
    monkeypatch.setenv("DGFEM_RESIDENT", "1")
    m = dg.box_mesh(2, 80, 3, jitter=0.1, seed=5)
    X = m.node_coords.reshape(-1, 3)
    u = np.zeros((4, len(X)))
    u[0] = np.exp(-(X ** 2).sum(1) / 0.1)
    solvers = [dg.Solver(m.node_coords, m.element_vertices, 3, None, rho0=RHO0, c0=C0, precision=dg.DG_MIXED)
               for _ in range(2)]
    dt = solvers[0].info().min_inradius / (C0 * 7)
    solvers[0].set_state(u)
    solvers[0].run_steps(300, dt)
    alone = solvers[0].get_state()
    out = [None, None]

    def work(k):
        for _ in range(3):
            solvers[k].set_state(u)
            solvers[k].run_steps(300, dt)
        out[k] = solvers[k].get_state()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    np.testing.assert_array_equal(out[0], alone)
    np.testing.assert_array_equal(out[1], alone)
