"""Which code runs a context's steps (dg_get_forms): the cases of the tests that compare the forms without
a DGFEM_KERNEL name with other kernels do run them, the resident loop hands no batch of theirs back, and
the default rules take each form on its side of the line."""
import numpy as np
import pytest

import dgfem_amd as dg
import test_gpu_quad
import test_gpu_resident
import test_gpu_tetmm

pytestmark = pytest.mark.gpu


@pytest.fixture
def forms(monkeypatch):
    """The forms of every solver that is closed, in order."""
    seen, close = [], dg.Solver.close

    def recording(self):
        if getattr(self, "_h", None):
            seen.append(self.forms())
        close(self)

    monkeypatch.setattr(dg.Solver, "close", recording)
    for name in ("DGFEM_KERNEL", "DGFEM_QUAD", "DGFEM_TET_MM", "DGFEM_POST_BRANCH", "DGFEM_RESIDENT",
                 "DGFEM_RESIDENT_PATIENCE"):
        monkeypatch.delenv(name, raising=False)
    return seen


@pytest.mark.parametrize("dim,order,fields,n", test_gpu_resident.CASES)
@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
@pytest.mark.parametrize("learned", [False, True])
def test_resident_cases_are_resident(dim, order, fields, n, precision, learned, forms, monkeypatch):
    """(The launches per stage they are compared with are not; FP64 grids with learned faces never are; one
    FP64 grid of order-2 tetrahedra has more blocks than the chip holds.)"""
    print(f"case forms resident dim={dim} order={order} fields={fields} n={n} precision={precision} learned={learned}",
          flush=True)
    m = dg.box_mesh(dim, n, order, jitter=0.1, seed=n)
    bc = dg.resolve_bc_sides(m, [(0x3, 1), (0x3C if dim == 3 else 0xC, 2 if learned else 0)])
    net = None
    if learned:
        net = dg.to_bf16(dg.closure_init(order + 1 if dim == 2 else dg.num_nodes(2, order), seed=4, out_scale=0.1, dim=dim))
    for resident in "10":
        test_gpu_resident._run(m, bc, order, fields, precision, resident, monkeypatch, steps=40, net=net)
    on, off = forms
    assert off.resident == 0 and off.resident_shape == -1 and off.resident_launches == 0
    if precision == dg.DG_FP64 and (learned or (dim, order, n) == (3, 2, 11)):
        assert on.resident == 0 and on.resident_launches == 0
    else:  # a batch ends at every save step, 0, 17 and 34
        assert on.resident == 1 and on.resident_shape >= 0 and on.resident_blocks > 0
        assert on.resident_launches == 3
    assert on.resident_aborts == 0 and off.resident_aborts == 0


def test_fallback_is_seen(forms, monkeypatch):
    print("case forms fallback", flush=True)
    test_gpu_resident.test_waiting_block_falls_back(dg.DG_MIXED, monkeypatch)
    assert [f.resident_aborts for f in forms] == [0, 1]
    assert [f.resident_launches for f in forms] == [0, 0]


@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
def test_no_second_attempt(precision, forms, monkeypatch):
    """Once a batch was handed back, neither the batches after it nor later runs of the context try the
    resident loop again; another context does."""
    print(f"case forms no second attempt precision={precision}", flush=True)
    m = dg.box_mesh(2, 20, 3, jitter=0.1, seed=3)
    u = np.zeros((4, m.K * m.Np))
    u[0] = np.exp(-(m.node_coords.reshape(-1, 3) ** 2).sum(1) / 0.1)
    states = []
    for patience in ("0", "2000000"):
        monkeypatch.setenv("DGFEM_RESIDENT_PATIENCE", patience)
        s = dg.Solver(m.node_coords, m.element_vertices, 3, None, rho0=1.225, c0=340.0, precision=precision)
        dt = s.info().min_inradius / (340.0 * 7)
        s.set_state(u)
        assert s.forms().resident == 1
        assert s.run(0.0, 39.5 * dt, dt, 9.5 * dt).steps == 40  # 4 batches and a rest
        f = s.forms()
        if patience == "0":
            assert (f.resident, f.resident_launches, f.resident_aborts) == (0, 0, 1)
            monkeypatch.delenv("DGFEM_RESIDENT_PATIENCE")
        else:
            assert f.resident == 1 and f.resident_launches >= 4 and f.resident_aborts == 0
        s.run_steps(20, dt)
        g = s.forms()
        assert g.resident == f.resident and g.resident_aborts == f.resident_aborts
        assert g.resident_launches == f.resident_launches + f.resident
        states.append(s.get_state())
        s.close()
    tol = test_gpu_resident.TOL[precision]
    assert 0 < np.linalg.norm(states[0]) and np.linalg.norm(states[0] - states[1]) <= tol * np.linalg.norm(states[1])


@pytest.mark.parametrize("integrator", [dg.DG_RK4, dg.DG_EULER])
def test_stage_form_cases(integrator, forms, monkeypatch):
    print(f"case forms stage integrator={integrator}", flush=True)
    test_gpu_quad.test_quad_equals_vm(3, "all", integrator, monkeypatch)
    monkeypatch.delenv("DGFEM_QUAD")
    for precision, order in ((dg.DG_FP64, 4), (dg.DG_FP64, 5), (dg.DG_MIXED, 4)):
        test_gpu_tetmm.test_matrix_core_equals_valu(order, 2, "both", 4, precision, integrator, monkeypatch)
    assert [f.stage_form for f in forms] == [dg.DG_FORM_KERNEL, dg.DG_FORM_QUAD] + 3 * [dg.DG_FORM_KERNEL, dg.DG_FORM_TET_MM]
    assert all(f.resident == 0 for f in forms)


@pytest.mark.parametrize("precision,order,n,form", [
    (dg.DG_FP64, 5, 6, dg.DG_FORM_KERNEL), (dg.DG_FP64, 5, 7, dg.DG_FORM_TET_MM),      # 1,296; 2,058
    (dg.DG_FP64, 4, 9, dg.DG_FORM_KERNEL), (dg.DG_FP64, 4, 10, dg.DG_FORM_TET_MM),     # 4,374; 6,000
    (dg.DG_MIXED, 4, 11, dg.DG_FORM_KERNEL), (dg.DG_MIXED, 4, 12, dg.DG_FORM_TET_MM),  # 7,986; 10,368
    (dg.DG_MIXED, 3, 30, dg.DG_FORM_KERNEL), (dg.DG_MIXED, 3, 31, dg.DG_FORM_QUAD),  # 162,000; 178,746
    (dg.DG_FP64, 3, 31, dg.DG_FORM_KERNEL), (dg.DG_MIXED, 5, 7, dg.DG_FORM_KERNEL)])
def test_default_rules(precision, order, n, form, forms):
    print(f"case forms rule precision={precision} order={order} n={n}", flush=True)
    m = dg.box_mesh(3, n, order)
    s = dg.Solver(m.node_coords, m.element_vertices, order, None, precision=precision)
    assert s.forms().stage_form == form
    assert s.forms().resident == 0
    s.close()


@pytest.mark.parametrize("fields", [4, 5])
@pytest.mark.parametrize("n,walls,shape", [(208, "rigid", 2), (222, "rigid", -1), (233, "rigid", -1), (222, "learned", 3)])
def test_order_1_triangles_at_5_blocks_per_cu(n, walls, shape, fields, forms):
    print(f"case forms order 1 n={n} walls={walls} fields={fields}", flush=True)
    m = dg.box_mesh(2, n, 1)
    bc = dg.resolve_bc_sides(m, [(0xF, dg.DG_BC_LEARNED if walls == "learned" else dg.DG_BC_REFLECTING)])
    s = dg.Solver(m.node_coords, m.element_vertices, 1, bc, fields=dg.DG_FIELDS_LEE5 if fields == 5 else dg.DG_FIELDS_REF4,
                  precision=dg.DG_MIXED)
    assert (s.forms().resident_shape, s.forms().resident) == (shape, int(shape >= 0))
    s.close()
