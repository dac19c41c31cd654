"""A smoother of the adjoint replaced between iterations by eigenvectors that do not separate by parity.
Its products pack undivided, at 96 points half again as large as the two parity classes of the other
smoothers, whose places in the fused iteration's operator array it must not touch.

Against a handle that had the same tensor from the start: the same operators and launches, so the same
bits.  Against the oracle to 1e-8: two eigen-decompositions of the other smoothers, whose solves agree to
1e-9, and differences of steps divided by 1e-2 on top of the fields' own size."""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu

NX, NY = 96, 97
ARGS = (NX, NY, 1e4, 1.0, 5e-3, 1.0, True)


def _start(g):
    g.set_temperature(0.5, 1.0, 1.0)
    g.set_velocity(0.5, 1.0, 1.0)


def _handle(o):
    from rustpde_amd import Navier2DAdjoint
    g = Navier2DAdjoint.new(*ARGS)
    g.set_temp_bc(o.fields.get("fieldbc"))
    g.navier.set_temp_bc(o.navier.get("fieldbc"))
    g.navier.set_tensor(3, *o.navier.tensor_setup(3))
    g.set_tensor(3, *o.fields.tensor_setup(3))
    _start(g)
    return g


def _state(g):
    return [f.vhat for f in (g.temp[0], g.ux[0], g.uy[0], g.pres[0], g.navier.pres[0])]


def _restore(g, state):
    for f, v in zip((g.temp[0], g.ux[0], g.uy[0], g.pres[0], g.navier.pres[0]), state):
        f.vhat = v


@pytest.mark.parametrize("slots", [(1,), (2,), (1, 2, 0)])
def test_smoother_replaced_between_iterations(oracle, slots):
    print("case smoothers replaced", slots, flush=True)
    o = oracle.NavierAdjoint.new(*ARGS)
    _start(o.fields)
    g, h = _handle(o), _handle(o)
    for s in slots:
        h.set_tensor(s, *o.smoother_tensor(s))
    start = _state(g)
    g.update(2)  # its own eigenvectors: parity classes, packed; then a replay
    for s in slots:  # one at a time, with iterations between
        g.set_tensor(s, *o.smoother_tensor(s))
        g.update(2)
    _restore(g, start)
    g.update(3)
    h.update(3)
    o.update(3)
    for name in ("temp", "ux", "uy"):
        for a, b in ((getattr(g, name)[0].vhat, getattr(h, name)[0].vhat),
                     (getattr(g, name)[1].vhat, getattr(h, name)[1].vhat),
                     (getattr(g, name)[1].unsmoothed, getattr(h, name)[1].unsmoothed)):
            assert np.array_equal(a, b), name
        assert rel_err(getattr(g, name)[0].vhat, o.fields.get(name)) < 1e-8, name
        assert rel_err(getattr(g, name)[1].vhat, o.residual(name)) < 1e-8, name
    g.close()
    h.close()
