"""Periodic steps whose convective terms are products with the dense x operators (small grids, and those
without fast transforms along one axis or both): even and odd row lengths, the y stage as products and (from 201
points of a fast length) as transforms, a fast x axis with a row length that has none.

Oracle tolerance 1e-12 after 5 steps, as the other periodic steps of these lengths; the single-precision
option has no kernels for the grids without fast transforms and leaves the step's bits as they are."""
import numpy as np
import pytest

from helpers import compare, init_pair, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [(12, 9), (22, 20), (30, 33), (34, 66), (64, 50), (36, 257), (100, 65), (256, 40), (64, 65), (256, 129), (512, 33), (128, 257)]


def _fields(g):
    return [f.vhat.copy() for f in (g.temp, g.ux, g.uy, g.pres[0])]


@pytest.mark.parametrize("shape", SHAPES)
def test_dense_periodic(oracle, shape):
    from rustpde_amd import Navier2D
    nx, ny = shape
    print("case periodic %dx%d, 5 steps" % shape, flush=True)
    make = lambda: Navier2D.new_periodic(nx, ny, 1e4, 1.0, 2e-3, 2.0)
    out = []
    for option in (None, "mixed", "batch", "solid"):
        g, o = make(), oracle.Navier2D.new_periodic(nx, ny, 1e4, 1.0, 2e-3, 2.0)
        init_pair(g, o, nx, ny, True, 1e-2, 3, "gaussian", velocity=(0.1, 2.0, 1.0))
        if option == "mixed":
            if shape in SHAPES[-4:]:  # FP32 transforms there
                g.close()
                continue
            g.set_option(g.OPT_MIXED, 1)
        if option == "batch":
            g.set_option(g.OPT_BATCH, 0)
        if option == "solid":
            g.solid = [np.zeros((nx, ny)), np.zeros((nx, ny))]
        g.update(5)
        if option is None:
            o.update(5)
            e = compare(g, o)
            for k in ("temp", "ux", "uy", "pres"):
                assert e[k] < 1e-12, (k, e)
            assert abs(g.eval_nu() - o.eval_nu()) < 1e-12 * abs(o.eval_nu())
        out.append(_fields(g))
        g.close()
    if len(out) == 4:
        assert all(np.array_equal(a, b) for a, b in zip(out[0], out.pop(1)))
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert rel_err(a, b) < 1e-12


@pytest.mark.parametrize("shape", [(32, 33), (64, 257), (128, 513)])
def test_rows_form_right_hand_sides(oracle, shape):
    """An aspect ratio that is no power of two (the division path of d/dx pres), with a pressure written
    between steps, rows of two and four entries a lane."""
    from rustpde_amd import Navier2D
    nx, ny = shape
    print("case periodic %dx%d, aspect 1.5" % shape, flush=True)
    g = Navier2D.new_periodic(nx, ny, 1e4, 1.0, 1e-3, 1.5)
    o = oracle.Navier2D.new_periodic(nx, ny, 1e4, 1.0, 1e-3, 1.5)
    init_pair(g, o, nx, ny, True, 1e-2, 3, "gaussian", velocity=(0.1, 2.0, 1.0))
    for _ in range(2):
        g.update(3)
        o.update(3)
        p = 0.5 * o.get("pres")
        g.pres[0].vhat = p
        o.set("pres", p)
    g.update(2)
    o.update(2)
    e = compare(g, o)
    for k in ("temp", "ux", "uy", "pres"):
        assert e[k] < 1e-12, (k, e)
    g.close()
