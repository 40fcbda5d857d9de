"""What a gradient leaves behind and starts its recomputation from: ql_adjoint_backward
returns the context to the final state of its forward, the record of the variable
steps and the drives included, and recomputes every segment from the record its
checkpoint holds.  Bars: bitwise where nothing but copies lies between, 1e-6 for
gradients against central differences."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = EPS = 1e-6


def _p(**kw):
    from ql_dns_amd.params import QLParams
    kw.setdefault("nu", 1 / 1500)
    kw.setdefault("eta", 1 / 1200)
    return QLParams(NX=8, NY=8, NZ=32, Ly=1.0, **kw)


def _start(p, lin, mf, kx0=None, t=0.0):
    from ql_dns_amd.capi import QLContext
    c = QLContext(p)
    c.set_state(lin, mf, kx0)
    c.linear_ops_init(t)
    return c


VARIABLE = [(0, 1), (1, 0), (2, 1), (2, 0)]


@pytest.mark.parametrize("model,integrator", VARIABLE)
def test_variable_steps_go_on_after_a_gradient_as_without_it(model, integrator):
    """The next step's size comes from the record of the forward's last step, not
    from one formed again with the drives of another segment."""
    from ql_dns_amd.ic import initial_state
    p = _p(model=model, integrator=integrator, dt=-0.05, CFL=1.0)
    lin, mf = initial_state(p, amp=0.05)
    out = []
    for grad in (False, True):
        c = _start(p, lin, mf)
        t = c.adjoint_forward(7, 3, 0.0)
        if grad:
            l, m, _ = c.get_state()
            c.adjoint_backward(1e-3 * l, m)
        cfl = c.calculate_cfl()
        dt = c.step(t)
        t = c.steps(3, t + dt)
        out.append((cfl, dt, t) + c.get_state())
        c.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_hd_variable_steps_adjoint_matches_frozen_step_differences():
    """HD_fullU's step size holds a source term of the drives above an energy cutoff
    (HD_fullU.cpp:614-624): the recomputed segments have to take the forward's steps.
    Central differences of the forward with its step sizes frozen."""
    from ql_dns_amd.ic import initial_state
    p = _p(model=2, dt=-0.05, CFL=1.0)
    n, every = 14, 5
    lin0, mf0 = initial_state(p, amp=0.05)
    alpha = 0.01 / float((np.abs(lin0) ** 2).sum())

    def loss(lin, mf):
        return 0.5 * float((np.abs(mf) ** 2).sum()) / p.NZ ** 2 + alpha * float((np.abs(lin) ** 2).sum())

    c = _start(p, lin0, mf0)
    t, dts = 0.0, []
    for _ in range(n):
        dts.append(c.step(t))
        t = t + dts[-1]
        c.remap(p.q * t)
    c.close()
    assert len(set(dts)) > 5, "the steps do not vary"

    def frozen(q, lin, mf):
        t, kx0 = 0.0, None
        for dt in dts:
            c = _start(q.replace(dt=float(dt)), lin, mf, kx0, t)
            c.step(t)
            t = t + dt
            c.remap(q.q * t)
            lin, mf, kx0 = c.get_state()
            c.close()
        return lin, mf

    c = _start(p, lin0, mf0)
    assert c.adjoint_forward(n, every, 0.0) == t
    linT, mfT, _ = c.get_state()
    gl0, gm0, gpar = c.adjoint_backward(2.0 * alpha * linT, mfT / p.NZ ** 2)
    c.close()
    lf, mff = frozen(p, lin0, mf0)
    assert rel_err(lf, linT) < 1e-13 and rel_err(mff, mfT) < 1e-13
    rng = np.random.default_rng(29)
    for d in range(2):
        vl = (rng.standard_normal(lin0.shape) + 1j * rng.standard_normal(lin0.shape)) * np.sqrt(np.mean(np.abs(lin0) ** 2))
        vl[::p.NY // 2, 0, 0] = 0
        vm = (rng.standard_normal(mf0.shape) + 1j * rng.standard_normal(mf0.shape)) * np.sqrt(np.mean(np.abs(mf0) ** 2))
        ad = float(np.sum(gl0.real * vl.real + gl0.imag * vl.imag) + np.sum(gm0.real * vm.real + gm0.imag * vm.imag))
        fd = (loss(*frozen(p, lin0 + EPS * vl, mf0 + EPS * vm)) -
              loss(*frozen(p, lin0 - EPS * vl, mf0 - EPS * vm))) / (2 * EPS)
        assert abs(ad - fd) <= TOL * abs(fd), f"state direction {d}: adjoint {ad!r} fd {fd!r}"
    for k, name in enumerate(("q", "omega", "nu")):
        h = EPS * abs(getattr(p, name))
        L = [loss(*frozen(p.replace(**{name: getattr(p, name) + s * h}), lin0, mf0)) for s in (1, -1)]
        fd = (L[0] - L[1]) / (2 * h)
        assert abs(gpar[k] - fd) <= TOL * abs(fd), f"d/d{name}: adjoint {gpar[k]!r} fd {fd!r}"


@pytest.mark.parametrize("model,integrator,dt", [(0, 1, 0.004), (1, 0, 0.004), (2, 1, 0.004), (0, 0, -0.05), (2, 1, -0.05)])
def test_drives_after_a_gradient_are_the_forwards(model, integrator, dt):
    """The drives and what the diagnostics read are those of the forward's last
    right-hand side, not of the segment recomputed last."""
    from ql_dns_amd.ic import initial_state
    p = _p(model=model, integrator=integrator, dt=dt, CFL=1.0)
    lin, mf = initial_state(p, amp=0.05)
    c = _start(p, lin, mf)
    t = c.adjoint_forward(7, 3, 0.0)
    want = (c.drive(), c.drive_real(), c.mf_real(), c.diagnostics(t), c.calculate_cfl())
    l, m, _ = c.get_state()
    c.adjoint_backward(1e-3 * l, m)
    got = (c.drive(), c.drive_real(), c.mf_real(), c.diagnostics(t), c.calculate_cfl())
    c.close()
    for a, b in zip(want, got):
        assert np.array_equal(a, b)
