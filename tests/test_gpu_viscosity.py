"""Hyperviscosity: the orders above 4 take |k|^order from pow (the exponent is the
integer order / 2, MHD_FullQlin.cpp:372), once per slot and time, in every mode
kernel.  Bars: the oracle to 1e-10 relative, as at the orders below; gradients
to 1e-6 of central differences."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _params(order, **kw):
    from ql_dns_amd.ic import mode_tables
    from ql_dns_amd.params import QLParams
    p = QLParams(viscosity_order=order, Ly=1.0, B0z=0.03, **kw)
    kx0, ky, _, _, kz, _ = mode_tables(p)
    k2 = np.abs(kx0).max() ** 2 + np.abs(ky).max() ** 2 + np.abs(kz).max() ** 2
    nu = 30.0 / k2 ** (order // 2)  # the largest wavenumbers decay over a few steps
    return p.replace(nu=nu, eta=1.3 * nu)


def _pair(p):
    from ql_dns_amd.capi import QLContext
    from ql_dns_amd.ic import initial_state
    from oracle.oracle import Oracle
    lin, mf = initial_state(p)
    o, g = Oracle.from_params(p, nthreads=8), QLContext(p)
    for x in (o, g):
        x.set_state(lin, mf)
        x.linear_ops_init(0.0)
    return o, g


@pytest.mark.parametrize("order", [5, 6, 8])
@pytest.mark.parametrize("integrator", [1, 0])
@pytest.mark.parametrize("NZ,line", [(32, 64), (32, 256), (64, 64), (64, 128), (128, 64), (128, 256), (256, 64), (256, 256)])
def test_steps_of_high_orders_match_oracle(order, integrator, NZ, line):
    p = _params(order, integrator=integrator, NX=8, NY=6, NZ=NZ)
    o, g = _pair(p)
    g.set_config(NZ, line, 64)
    ro, rg = o.rhs(0.1, 0.01), g.rhs(0.1, 0.01)
    for a, b in zip(rg, ro):
        assert rel_err(a, b) < TOL
    assert g.steps(12, 0.0) == o.steps(12, 0.0)
    (lo, mo, ko), (lg, mg, kg) = o.get_state(), g.get_state()
    assert np.array_equal(kg, ko)
    assert rel_err(mg, mo) < TOL and rel_err(lg, lo) < TOL


@pytest.mark.parametrize("integrator,NZ", [(1, 32), (0, 64), (0, 128)])
def test_gradients_of_high_orders_match_finite_differences(integrator, NZ):
    from ql_dns_amd.adjoint import mf_energy
    from ql_dns_amd.capi import QLContext
    from ql_dns_amd.ic import initial_state
    p = _params(6, integrator=integrator, NX=8, NY=8, NZ=NZ)
    # the small scales, which the viscosity acts on, hold as much as the large ones:
    # else the loss depends on it by less than differences resolve
    lin, mf = initial_state(p, kdecay=1e5)
    alpha = 0.01 / float((np.abs(lin) ** 2).sum())

    def run(q, grad=False):
        c = QLContext(q)
        c.set_state(lin, mf)
        c.linear_ops_init(0.0)
        c.adjoint_forward(8, 3, 0.0)
        l, m, _ = c.get_state()
        L = mf_energy(q, m) + alpha * float((np.abs(l) ** 2).sum())
        if grad:
            g_mf = np.zeros_like(m)
            g_mf[:2] = m[:2] / q.NZ ** 2
            L = c.adjoint_backward(2 * alpha * l, g_mf)[2]
        c.close()
        return L

    g = run(p, True)
    for k, name in enumerate(("q", "omega", "nu", "eta")):
        h = 1e-6 * getattr(p, name)
        fd = (run(p.replace(**{name: getattr(p, name) + h})) - run(p.replace(**{name: getattr(p, name) - h}))) / (2 * h)
        assert abs(g[k] - fd) <= 1e-6 * abs(fd), f"d/d{name}: adjoint {g[k]!r} fd {fd!r}"
