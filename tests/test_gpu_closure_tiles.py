"""Exterior states of learned faces in tiles of 16 (mixed precision; FP64: 4 faces per wave): face
counts around a tile's edge, every network shape and both field counts, the right-hand side against
the NumPy restatement with the oracle's exterior states (bars as in test_gpu_closure.py)."""
import numpy as np
import pytest

import closure_oracle as co
import dgfem_amd as dg
import nodal_ref
from cases import rel_l2, smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,bar", [(dg.DG_FP64, 1e-6), (dg.DG_MIXED, 2e-5)])
@pytest.mark.parametrize("faces", [1, 15, 16, 17, 48])
@pytest.mark.parametrize("dim,order,fields", [(2, 1, 4), (2, 2, 5), (2, 3, 4), (2, 4, 4), (2, 5, 5), (3, 1, 5), (3, 2, 4),
                                              (3, 3, 4)])
def test_face_counts(dim, order, fields, faces, precision, bar):
    print(f"case closure tiles dim={dim} order={order} fields={fields} faces={faces} precision={precision}", flush=True)
    v0, rho0, c0 = (40.0, -25.0, 10.0 if dim == 3 else 0.0), 1.225, 100.0
    m = dg.box_mesh(dim, 13 if dim == 2 else 3, order, jitter=0.1, seed=faces)
    flat = np.flatnonzero(m.face_side.reshape(-1) >= 0)
    assert flat.size >= faces
    bc = np.zeros(m.face_side.size, dtype=np.int8)
    bc[np.random.default_rng(faces).choice(flat, faces, replace=False)] = dg.DG_BC_LEARNED
    bc = bc.reshape(m.face_side.shape)
    nfp = order + 1 if dim == 2 else dg.num_nodes(2, order)
    bits = dg.to_bf16(np.random.default_rng(7).normal(0, 0.2, dg.closure_num_params(nfp, dim)).astype(np.float32))
    s = dg.Solver(m.node_coords, m.element_vertices, order, bc, v0=v0, rho0=rho0, c0=c0, precision=precision,
                  fields=dg.DG_FIELDS_LEE5 if fields == 5 else dg.DG_FIELDS_REF4)
    assert s.learned_faces()[0].size == faces
    s.set_closure(bits)
    u = smooth_state(m)
    if fields == 5:
        u = np.concatenate([u, u[:1] / c0 ** 2])
    k = s.rhs(u, 1e-5)
    pre = dg.mesh_precompute(m.node_coords, m.element_vertices, order, bc)
    ops = dg.ref_operators(dim, order)

    def exterior(qm, n):
        ext = np.zeros_like(qm)
        ext[..., :4] = co.exterior(qm[..., :4], n, co.bf16_to_f64(bits), v0, rho0, c0, dim=dim)
        if fields == 5:
            ext[..., 4] = qm[..., 4] + (ext[..., 0] - qm[..., 0]) / c0 ** 2
        return ext

    kr = nodal_ref.nodal_rhs(u, pre, ops, dim, v0, rho0, c0, 1e-5, nf=fields, closure=exterior)
    for f in range(fields):
        if np.abs(kr[f]).max() > 0:
            assert rel_l2(k[f], kr[f]) < bar, (f, rel_l2(k[f], kr[f]))
    s.close()
