"""The fused adjoint iteration (three fields per launch, rows of the right-hand sides, graph replays) at
the edges of its kernels: odd and even lengths around multiples of 16 points, a periodic grid without
fast transforms, temperature on the Dirichlet and the Neumann basis, fields and set-up written between
iterations.

After 4 iterations the fields agree with the oracle to 1e-11: an iteration divides differences of steps
by dt = 1e-2 and takes second derivatives, so the 1e-12 of single steps is near rounding."""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


def _pair(oracle, periodic, nx, ny, adiabatic=True):
    from rustpde_amd import Navier2DAdjoint
    if periodic:
        args = (nx, ny, 1e4, 1.0, 5e-3, 2.0)
        g, o = Navier2DAdjoint.new_periodic(*args), oracle.NavierAdjoint.new_periodic(*args)
    else:
        args = (nx, ny, 1e4, 1.0, 5e-3, 1.0, adiabatic)
        g, o = Navier2DAdjoint.new(*args), oracle.NavierAdjoint.new(*args)
        g.set_temp_bc(o.fields.get("fieldbc"))
        g.navier.set_temp_bc(o.navier.get("fieldbc"))
        g.navier.set_tensor(3, *o.navier.tensor_setup(3))
        g.set_tensor(3, *o.fields.tensor_setup(3))
        for s in range(3):
            g.set_tensor(s, *o.smoother_tensor(s))
    for x in (g, o.fields):
        x.set_temperature(0.5, 1.0, 1.0)
        x.set_velocity(0.5, 1.0, 1.0)
    return g, o


def _compare(g, o, tol):
    for name in ("temp", "ux", "uy"):
        assert rel_err(getattr(g, name)[0].vhat, o.fields.get(name)) < tol, name
        assert rel_err(getattr(g, name)[1].vhat, o.residual(name)) < tol, name
        assert rel_err(getattr(g, name)[1].unsmoothed, o.unsmoothed(name)) < tol, name
    assert rel_err(g.pres[0].vhat, o.fields.get("pres")) < tol
    assert np.abs(g.norms() - o.norms()).max() < tol * np.abs(o.norms()).max()


@pytest.mark.parametrize("case", [(False, 10, 12, True), (False, 17, 16, True), (False, 33, 34, False),
                                  (False, 50, 35, True), (True, 16, 17), (True, 12, 9), (True, 36, 40), (True, 64, 33)])
def test_fused_adjoint(oracle, case):
    print("case fused adjoint", case, flush=True)
    g, o = _pair(oracle, *case)
    g.update(4)
    o.update(4)
    _compare(g, o, 1e-11)
    assert abs(g.get_time() - o.get_time()) < 1e-12
    # a field written between iterations and a new boundary field take effect on the replays
    t = 0.5 * o.fields.get("temp")
    g.temp[0].vhat = t
    g.set_temp_bc(o.fields.get("fieldbc"))
    o.fields.set("temp", t)
    g.update(1)
    g.update(2)
    o.update(3)
    _compare(g, o, 1e-11)
    g.close()


def test_replays_match_single_iterations():
    """The product's own eigenvectors (parity classes): six iterations of one call and six calls with a
    field written back between them hold the same bits."""
    from rustpde_amd import Navier2DAdjoint
    out = []
    for one in (True, False):
        g = Navier2DAdjoint.new(40, 41, 1e4, 1.0, 5e-3, 1.0, True)
        g.set_temperature(0.5, 1.0, 1.0)
        g.set_velocity(0.5, 1.0, 1.0)
        if one:
            g.update(6)
        else:
            for _ in range(6):
                g.update(1)
                g.ux[0].vhat = g.ux[0].vhat
        out.append([f[0].vhat for f in (g.temp, g.ux, g.uy, g.pres)])
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
