"""The caller's state in and out of the device layout: every (dim, order, fields) and precision, an
element count that leaves a partial last block, and elements whose nodes after the vertices come in
an order of their own. FP64 comes back bit for bit; mixed precision as the sum of the nearest FP32
value and the FP32 value nearest the remainder (zeros of either sign, infinities and NaN included)."""
import numpy as np
import pytest

import dgfem_amd as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,order,fields", [(2, 1, 4), (2, 3, 5), (2, 5, 4), (3, 1, 5), (3, 2, 4), (3, 3, 4), (3, 4, 5),
                                              (3, 5, 5)])
@pytest.mark.parametrize("precision", [dg.DG_FP64, dg.DG_MIXED])
def test_state_round_trip(dim, order, fields, precision):
    print(f"case state round trip dim={dim} order={order} fields={fields} precision={precision}", flush=True)
    m = dg.box_mesh(dim, 3, order, jitter=0.1, seed=4)
    rng = np.random.default_rng(order)
    X = m.node_coords.copy()
    for e in range(m.K):  # an own node order per element, the vertices first
        X[e, dim + 1:] = X[e, dim + 1 + rng.permutation(m.Np - dim - 1)]
    s = dg.Solver(X, m.element_vertices, order, None, rho0=1.2, c0=300.0,
                  fields=dg.DG_FIELDS_LEE5 if fields == 5 else dg.DG_FIELDS_REF4, precision=precision)
    u = rng.normal(size=s.state_shape) * 10.0 ** rng.integers(-30, 30, s.state_shape)
    u[:, :5] = 0.0
    u[:, 5] = -0.0
    u[0, 6], u[1, 6], u[2, 6] = np.inf, -np.inf, np.nan
    s.set_state(u)
    got = s.get_state()
    if precision == dg.DG_MIXED:
        with np.errstate(invalid="ignore"):
            hi = u.astype(np.float32)
            u = hi.astype(np.float64) + (u - hi).astype(np.float32).astype(np.float64)
    np.testing.assert_array_equal(got, u)
    # the layout itself: the initial condition is evaluated node by node on the host
    s.set_state(np.zeros_like(u))
    s.add_gaussian(0.1, -0.2, 0.3 if dim == 3 else 0.0, 0.2, 1.5)
    x = X.reshape(-1, 3) - np.array([0.1, -0.2, 0.3 if dim == 3 else 0.0])
    want = 1.5 * np.exp(-(x ** 2).sum(1) / 0.2)
    np.testing.assert_allclose(s.get_state()[0], want, rtol=1e-13 if precision == dg.DG_FP64 else 1e-7)
    s.close()
